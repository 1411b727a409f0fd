// Decode-step kernels: single-query attention (split over the cache with an
// in-kernel merge) and the bandwidth-trivial ops a KV-cached step needs.
// References: shaders/single_query_attention.comp:26-72, rms_norm.comp:21-49,
// rope.comp:18-41, gelu.comp:15-30, add.comp:18-26, embed.comp:18-28,
// greedy_sample.comp:24-64.
#include "kernels.h"

#include <math.h>

#include <algorithm>
#include <cmath>

namespace evkhip {

namespace {

// ---------------------------------------------------------------------------
// Single-query attention.  Grid (heads, nsplit); 256 threads.  A workgroup
// covers cache rows [split*chunk, +chunk) of one head: LPK = DH/8 lanes per
// key (16 bytes each), 256/LPK keys per pass, U passes requested at once and
// the next U while those are scored (U = 1 where a split is one pass).
// Latency bounds a short cache and the bytes in flight a long one; with one
// pass at a time and a fence per workgroup, us before -> now, the step's two
// cache writes included: 16 caches of 160 rows of 256 14.3 -> 9.8, 38 of 739
// 56 -> 12, one of 4000 rows of 12 heads of 64 62 -> 11, 32 of 2001 rows of 8
// heads of 128 121 -> 47 (5.5 TB/s).  Partial (m, l, o) go to workspace at agent scope; the last
// workgroup of a head merges the splits in split order, every partial it
// needs requested in batches of SQ_MB.
// ---------------------------------------------------------------------------
constexpr int SQ_U = 4, SQ_MB = 16;
constexpr int SQ_SPLITS = 256;  // at most: one thread each in the merge
struct SqArgs {
    const f16* q;
    const f16* kc;
    const f16* vc;
    f16* out;
    int64_t row_stride;  // elements between consecutive cache rows
    int64_t cache_bstride;  // elements between the caches of consecutive sequences
    int heads, L, chunk;    // heads per sequence; grid.x = sequences * heads
    float scale_log2;
    float* part;         // [heads][nsplit][2 + DH]
    unsigned* counters;  // [heads]
};

constexpr float kLog2e = 1.4426950408889634f;

template <int DH, int U>
__global__ __launch_bounds__(256) void sq_attention(SqArgs a) {
    constexpr int LPK = DH / 8;             // lanes per key
    constexpr int KPP = 256 / LPK;          // keys per pass
    static_assert(KPP >= 4, "at least one key slot per wave");
    __shared__ float s_m[4], s_w[4];
    __shared__ float s_o[4][DH];
    // h: (sequence, head) pair; q, out and the workspace are indexed by it,
    // the caches by the sequence's cache and the head's columns
    const int h = blockIdx.x, split = blockIdx.y, nsplit = gridDim.y;
    const int seq = h / a.heads, hc = h - seq * a.heads;
    const f16* kc = a.kc + (int64_t)seq * a.cache_bstride + (int64_t)hc * DH;
    const f16* vc = a.vc + (int64_t)seq * a.cache_bstride + (int64_t)hc * DH;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int sub = tid % LPK, kslot = tid / LPK;
    const int j0 = split * a.chunk, j1 = min(a.L, j0 + a.chunk);

    float qv[8];
    {
        half8 qh = *reinterpret_cast<const half8*>(a.q + (int64_t)h * DH + sub * 8);
#pragma unroll
        for (int e = 0; e < 8; ++e) qv[e] = (float)qh[e];
    }
    float m = -INFINITY, l = 0.0f, o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = 0.0f;

    auto load = [&](int jb, half8 (&k)[U], half8 (&v)[U]) {  // rows past the range: its last one, masked below
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t at = (int64_t)min(jb + u * KPP + kslot, j1 - 1) * a.row_stride + sub * 8;
            k[u] = *reinterpret_cast<const half8*>(kc + at);
            v[u] = *reinterpret_cast<const half8*>(vc + at);
        }
    };
    half8 kh[U], vh[U];
    if (j0 < j1) load(j0, kh, vh);
    for (int jb = j0; jb < j1; jb += KPP * U) {
        half8 kn[U], vn[U];
        const bool more = jb + KPP * U < j1;
        if (more) {
            load(jb + KPP * U, kn, vn);
        } else {  // weight 0 times the last row again is not 0 where that row holds an infinity
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (jb + u * KPP + kslot >= j1) vh[u] = half8{};
        }
        // online softmax per lane group (all LPK lanes of a key hold the same s)
        float s[U], mn = m;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float d = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) d += qv[e] * (float)kh[u][e];
            d = lanes_sum<LPK>(d);
            s[u] = jb + u * KPP + kslot < j1 ? d * a.scale_log2 : -INFINITY;
            mn = fmaxf(mn, s[u]);
        }
        const float base = mn == -INFINITY ? 0.0f : mn;
        const float al = exp2f(m - base);
        l *= al;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] *= al;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float pe = exp2f(s[u] - base);
            l += pe;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] += pe * (float)vh[u][e];
        }
        m = mn;
        if (more) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                kh[u] = kn[u];
                vh[u] = vn[u];
            }
        }
    }
    // Merge the key slots of the workgroup: within a wave (slots sharing sub)
    // then across waves through LDS.
#pragma unroll
    for (int off = LPK; off < 64; off <<= 1) {
        float m2 = __shfl_xor(m, off, 64), l2 = __shfl_xor(l, off, 64);
        float mn = fmaxf(m, m2);
        float base = mn == -INFINITY ? 0.0f : mn;
        float a1 = exp2f(m - base), a2 = exp2f(m2 - base);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = o[e] * a1 + __shfl_xor(o[e], off, 64) * a2;
        l = l * a1 + l2 * a2;
        m = mn;
    }
    if (lane < LPK) {
        if (sub == 0) { s_m[wave] = m; s_w[wave] = l; }
#pragma unroll
        for (int e = 0; e < 8; ++e) s_o[wave][sub * 8 + e] = o[e];
    }
    __syncthreads();
    float* part = a.part + ((int64_t)h * nsplit + split) * (2 + DH);
    if (tid < DH) {
        float mm = fmaxf(fmaxf(s_m[0], s_m[1]), fmaxf(s_m[2], s_m[3]));
        float base = mm == -INFINITY ? 0.0f : mm;
        float ll = 0.0f, oo = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            float f = exp2f(s_m[w] - base);
            ll += s_w[w] * f;
            oo += s_o[w][tid] * f;
        }
        if (nsplit == 1) {
            a.out[(int64_t)h * DH + tid] = (f16)(ll > 0.0f ? oo / ll : 0.0f);
        } else {
            st_ag(part + 2 + tid, oo);
            if (tid == 0) {
                st_ag(part, mm);
                st_ag(part + 1, ll);
            }
        }
    }
    if (nsplit == 1 || !arrive_last(a.counters + h, nsplit)) return;
    // Weights of the splits, one thread each; then GR groups of DH threads sum
    // every GR-th split's o and meet in LDS in group order.
    constexpr int GR = 256 / DH;
    __shared__ float s_wt[SQ_SPLITS], s_sum[GR][DH];
    const float* ph = a.part + (int64_t)h * nsplit * (2 + DH);
    const float m_sp = tid < nsplit ? ld_ag(ph + tid * (2 + DH)) : -INFINITY;
    const float l_sp = tid < nsplit ? ld_ag(ph + tid * (2 + DH) + 1) : 0.0f;
    float mm = wave_max(m_sp);
    if (lane == 0) s_m[wave] = mm;
    __syncthreads();
    mm = fmaxf(fmaxf(s_m[0], s_m[1]), fmaxf(s_m[2], s_m[3]));
    const float wt = exp2f(m_sp - (mm == -INFINITY ? 0.0f : mm));
    const float lw = wave_sum(l_sp * wt);
    s_wt[tid] = wt;
    if (lane == 0) s_w[wave] = lw;
    __syncthreads();
    const float ll = s_w[0] + s_w[1] + s_w[2] + s_w[3];
    const int gr = tid / DH, dim = tid % DH;
    float oo = 0.0f;
    for (int sp = gr; sp < nsplit; sp += GR * SQ_MB) {
        float t[SQ_MB];
#pragma unroll
        for (int u = 0; u < SQ_MB; ++u) t[u] = sp + u * GR < nsplit ? ld_ag(ph + (sp + u * GR) * (2 + DH) + 2 + dim) : 0.0f;
#pragma unroll
        for (int u = 0; u < SQ_MB; ++u) oo += t[u] * (sp + u * GR < nsplit ? s_wt[sp + u * GR] : 0.0f);
    }
    s_sum[gr][dim] = oo;
    __syncthreads();
    if (tid < DH) {
        oo = 0.0f;
#pragma unroll
        for (int g = 0; g < GR; ++g) oo += s_sum[g][tid];
        a.out[(int64_t)h * DH + tid] = (f16)(ll > 0.0f ? oo / ll : 0.0f);
    }
}

// Any head size: one workgroup per head, the shader's algorithm with the
// softmax and the P.V product spread over the workgroup.
__global__ __launch_bounds__(256) void sq_attention_scalar(SqArgs a, int dh) {
    extern __shared__ float sh[];  // scores[L] then q[dh]
    float* sc = sh;
    float* qs = sh + a.L;
    __shared__ float s_red[256];
    const int h = blockIdx.x, tid = threadIdx.x;
    const int seq = h / a.heads, hc = h - seq * a.heads;
    const f16* kc = a.kc + (int64_t)seq * a.cache_bstride + (int64_t)hc * dh;
    const f16* vc = a.vc + (int64_t)seq * a.cache_bstride + (int64_t)hc * dh;
    for (int d = tid; d < dh; d += 256) qs[d] = (float)a.q[(int64_t)h * dh + d];
    __syncthreads();
    const float inv = a.scale_log2;
    float mx = -INFINITY;
    for (int j = tid; j < a.L; j += 256) {
        const f16* kr = kc + (int64_t)j * a.row_stride;
        float s = 0.0f;
        for (int d = 0; d < dh; ++d) s += qs[d] * (float)kr[d];
        sc[j] = s * inv;
        mx = fmaxf(mx, sc[j]);
    }
    s_red[tid] = mx;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) s_red[tid] = fmaxf(s_red[tid], s_red[tid + o]);
        __syncthreads();
    }
    mx = s_red[0];
    __syncthreads();
    float sum = 0.0f;
    for (int j = tid; j < a.L; j += 256) {
        sc[j] = exp2f(sc[j] - mx);
        sum += sc[j];
    }
    s_red[tid] = sum;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) s_red[tid] += s_red[tid + o];
        __syncthreads();
    }
    const float is = s_red[0] > 0.0f ? 1.0f / s_red[0] : 0.0f;
    for (int d = tid; d < dh; d += 256) {
        float acc = 0.0f;
        for (int j = 0; j < a.L; ++j) acc += sc[j] * (float)vc[(int64_t)j * a.row_stride + d];
        a.out[(int64_t)h * dh + d] = (f16)(acc * is);
    }
}

// ---------------------------------------------------------------------------
// KV-cache append: rows [pos0, pos0 + n) of each sequence's cache (max_seq, D)
// take the rows of src (batch, n, D).  One thread per 8 values (16 bytes)
// when D % 8 == 0 and both buffers are 16-byte aligned, else per value.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void kv_write_k(const f16* src, f16* cache, int64_t total, int n, int D,
                                                  int max_seq, int pos0, int vec) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int W = vec ? 8 : 1;
    const int64_t e0 = i * W;  // element index in src
    if (e0 >= total) return;
    const int64_t row = e0 / D, col = e0 % D;
    const int64_t b = row / n, r = row % n;
    f16* dst = cache + (b * max_seq + pos0 + r) * D + col;
    if (vec) *reinterpret_cast<u32x4*>(dst) = *reinterpret_cast<const u32x4*>(src + e0);
    else *dst = src[e0];
}

// ---------------------------------------------------------------------------
// rms_norm: one wave per row, 4 rows per workgroup.  Rows of D <= 512 * NV
// whose length is a multiple of 8 stay in registers (16-byte accesses at any
// alignment, one read and one write of each value); longer or odd rows are
// walked element by element, twice.  Launch-bound at 1000 rows of 768: 3.4 us
// (walked, 2-byte accesses: 7.7).
// ---------------------------------------------------------------------------
DEV float clamp_f16(float v) { return fminf(fmaxf(v, -65504.0f), 65504.0f); }

template <int NV>
__global__ __launch_bounds__(256) void rms_norm_reg_k(const f16* in, f16* out, int64_t rows, int D, float eps) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= rows) return;
    const f16* x = in + row * D;
    half8 r[NV];
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int c = (lane + 64 * u) * 8;
        r[u] = half8{};
        if (c < D) r[u] = ld_h8(x + c);
    }
    float ss = 0.0f;
#pragma unroll
    for (int u = 0; u < NV; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float v = clamp_f16((float)r[u][e]);
            ss += v * v;
        }
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)D + eps);
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int c = (lane + 64 * u) * 8;
        if (c >= D) continue;
        half8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (f16)(clamp_f16((float)r[u][e]) * inv);
        st_h8(out + row * D + c, o);
    }
}

__global__ __launch_bounds__(256) void rms_norm_k(const f16* in, f16* out, int64_t rows, int D, float eps) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= rows) return;
    const f16* x = in + row * D;
    float ss = 0.0f;
    for (int j = lane; j < D; j += 64) {
        const float v = clamp_f16((float)x[j]);
        ss += v * v;
    }
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)D + eps);
    for (int j = lane; j < D; j += 64) out[row * D + j] = (f16)(clamp_f16((float)x[j]) * inv);
}

// rope: one thread per rotated pair.
__global__ __launch_bounds__(256) void rope_k(const f16* in, f16* out, int B, int S, int E, float base,
                                               int pos0, int hd) {
    const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int pairs = E / 2;
    if (gid >= (int64_t)B * S * pairs) return;
    const int pr = (int)(gid % pairs);
    const int64_t tmp = gid / pairs;
    const int t = (int)(tmp % S);
    const int64_t idx = tmp * E + 2 * pr;
    const int pp = pr % (hd / 2);
    const float x0 = (float)in[idx], x1 = (float)in[idx + 1];
    const float inv_freq = powf(base, -2.0f * (float)pp / (float)hd);
    const float ang = (float)(pos0 + t) * inv_freq;
    float s, c;
    sincosf(ang, &s, &c);
    out[idx] = (f16)(x0 * c - x1 * s);
    out[idx + 1] = (f16)(x0 * s + x1 * c);
}


// Elementwise: 8 consecutive values per thread in 16-byte accesses (at any
// alignment), the last thread value by value.  Memory-bound: gelu over 2560 x
// 3072 7.7 us = 4.1 TB/s (19.2 us with one value per thread and tanhf).
template <class F>
DEV void each8(int64_t n, F&& f) {
    const int64_t i0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (i0 < n) f(i0, n - i0 < 8 ? (int)(n - i0) : 8);
}
DEV half8 ld_n(const f16* p, int n) {
    if (n == 8) return ld_h8(p);
    half8 v = {};
    if (n > 0) {  // the last value again past the end: no branch, hence no wait, between the loads
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = p[min(e, n - 1)];
    }
    return v;
}
DEV void st_n(f16* p, const half8& v, int n) {
    if (n == 8) return st_h8(p, v);
#pragma unroll
    for (int e = 0; e < 7; ++e)
        if (e < n) p[e] = v[e];
}

__global__ __launch_bounds__(256) void gelu_k(const f16* in, f16* out, int64_t n) {
    each8(n, [&](int64_t i, int k) {
        half8 v = ld_n(in + i, k);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (f16)gelu_fast((float)v[e]);
        st_n(out + i, v, k);
    });
}

__global__ __launch_bounds__(256) void add_k(const f16* a, const f16* b, f16* c, int64_t n) {
    each8(n, [&](int64_t i, int k) {
        const half8 x = ld_n(a + i, k), y = ld_n(b + i, k);
        half8 v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (f16)((float)x[e] + (float)y[e]);
        st_n(c + i, v, k);
    });
}

// One thread per W values of a row (W = 8 or 1; dim / W rounded up pieces a row).
template <int W>
__global__ __launch_bounds__(256) void embed_k(const f16* table, const uint16_t* idx, f16* out, int64_t n_idx,
                                                int dim, int pieces, int vocab) {
    const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (gid >= n_idx * pieces) return;
    const int64_t i = gid / pieces;
    const int d = (int)(gid % pieces) * W;
    const int tok = min((int)idx[i], vocab - 1);
    const f16* src = table + (int64_t)tok * dim + d;
    f16* dst = out + i * dim + d;
    if constexpr (W == 1) {
        *dst = *src;
    } else {
        const int k = min(8, dim - d);
        st_n(dst, ld_n(src, k), k);
    }
}

// ---------------------------------------------------------------------------
// greedy_sample.  The shader's winner is the maximum under the total order
// (value desc, bitrev8(j mod 256) asc, j asc) over valid candidates
// (value > -FLT_MAX), j = token - token_base; with no valid candidate it is
// token_base.  Any reduction tree over this order gives the same winner.
// ---------------------------------------------------------------------------

// One workgroup of NT threads per sequence; a thread requests LD pieces of W
// values (8 or 1) before it looks at any; the row may start at any fp16
// address.  greedy_launch chooses.
template <int NT, int W, int LD>
__global__ __launch_bounds__(NT) void greedy_k(const f16* logits, uint16_t* out, int S, int V, int position,
                                                int token_base, int token_count) {
    __shared__ float s_v[NT / 64];
    __shared__ uint32_t s_r[NT / 64];
    const int b = blockIdx.x, tid = threadIdx.x;
    const f16* row = logits + ((int64_t)b * S + position) * V + token_base;
    float bv = -3.402823466e+38f;
    uint32_t br = 0u;  // rank of j = 0 (token_base)
    for (int j0 = tid * W; j0 < token_count; j0 += NT * W * LD) {
        half8 v[LD];
#pragma unroll
        for (int u = 0; u < LD; ++u) {
            const int j = j0 + u * NT * W;
            if constexpr (W == 8) v[u] = ld_n(row + j, max(0, min(8, token_count - j)));
            else v[u][0] = row[min(j, token_count - 1)];
        }
#pragma unroll
        for (int u = 0; u < LD; ++u)
#pragma unroll
            for (int e = 0; e < W; ++e) {
                const int j = j0 + u * NT * W + e;
                const float x = (float)v[u][e];
                const uint32_t r = greedy_rank((uint32_t)j);
                if (j < token_count && x > -3.402823466e+38f && greedy_better(x, r, bv, br)) {
                    bv = x;
                    br = r;
                }
            }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        float v2 = __shfl_xor(bv, o, 64);
        uint32_t r2 = __shfl_xor(br, o, 64);
        if (greedy_better(v2, r2, bv, br)) { bv = v2; br = r2; }
    }
    if ((tid & 63) == 0) { s_v[tid >> 6] = bv; s_r[tid >> 6] = br; }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < NT / 64; ++w)
            if (greedy_better(s_v[w], s_r[w], bv, br)) { bv = s_v[w]; br = s_r[w]; }
        out[b] = (uint16_t)(token_base + greedy_index(br));
    }
}

// Decode-attention workspace (grow-only).
float* g_sq_part = nullptr;
size_t g_sq_part_elems = 0;
unsigned* g_sq_cnt = nullptr;
size_t g_sq_cnt_n = 0;

}  // namespace

void decode_ops_free_workspace() {
    if (g_sq_part) (void)hipFree(g_sq_part);
    if (g_sq_cnt) (void)hipFree(g_sq_cnt);
    g_sq_part = nullptr;
    g_sq_cnt = nullptr;
    g_sq_part_elems = g_sq_cnt_n = 0;
}

int sq_attention_launch(const f16* q, const f16* kc, const f16* vc, f16* out, int64_t row_stride, int heads,
                        int dh, int L, bool vec_ok, hipStream_t st, int batch, int64_t cache_bstride) {
    SqArgs a{};
    a.q = q; a.kc = kc; a.vc = vc; a.out = out;
    a.row_stride = row_stride; a.heads = heads; a.L = L;
    a.cache_bstride = cache_bstride;
    // from here on `heads` counts (sequence, head) pairs: one grid row each
    heads *= batch;
    a.scale_log2 = (1.0f / sqrtf((float)dh)) * kLog2e;
    const bool vec = vec_ok && (dh == 16 || dh == 32 || dh == 64 || dh == 128 || dh == 256) && (row_stride % 8 == 0);
    if (!vec) {
        size_t shm = sizeof(float) * ((size_t)L + dh);
        if (shm > 64 * 1024)
            return set_error(EVKHIP_ERR_UNSUPPORTED, "single_query_attention: head size %d with %d cached rows "
                             "needs the vector path (dh in {16,32,64,128,256})", dh, L);
        hipLaunchKernelGGL(sq_attention_scalar, dim3(heads), dim3(256), shm, st, a, dh);
        hipError_t e = hipGetLastError();
        return e == hipSuccess ? EVKHIP_OK : check_hip(e, "sq_attention_scalar launch");
    }
    // A split walks `step` rows at a time (about a microsecond each), and the
    // merge takes about as long per SQ_MB splits: chunk / step + splits / SQ_MB
    // is least at splits = sqrt(SQ_MB L / step), within two workgroups per CU.
    // Over 58 drawn calls (L to 20000, head sizes 16 to 256, up to 128 caches)
    // 0.66 of the time of 64 rows a split and one pass in flight, geometric mean.
    const int cus = device_cu_count();
    int nsplit = 1, chunk = std::max(L, 1);
    const int step = 256 / (dh / 8) * SQ_U;
    if (L > std::max(step, 64)) {  // up to 64 rows: no workspace
        const int few = (int)std::ceil(std::sqrt((double)SQ_MB * L / step));
        nsplit = std::max(1, std::min({(L + step - 1) / step, (2 * cus + heads - 1) / heads, few, SQ_SPLITS}));
        chunk = ((L + nsplit - 1) / nsplit + step - 1) / step * step;  // whole steps
        nsplit = (L + chunk - 1) / chunk;
    }
    a.chunk = chunk;
    if (nsplit > 1) {
        size_t need = (size_t)heads * nsplit * (2 + dh);
        if (need > g_sq_part_elems) {
            if (g_sq_part) EVK_HIP(hipFree(g_sq_part));
            // a failed allocation below leaves an empty workspace, never a
            // stale size over a null pointer
            g_sq_part = nullptr;
            g_sq_part_elems = 0;
            EVK_HIP(hipMalloc(&g_sq_part, need * sizeof(float)));
            g_sq_part_elems = need;
        }
        if ((size_t)heads > g_sq_cnt_n) {
            if (g_sq_cnt) EVK_HIP(hipFree(g_sq_cnt));
            g_sq_cnt = nullptr;
            g_sq_cnt_n = 0;
            EVK_HIP(hipMalloc(&g_sq_cnt, heads * sizeof(unsigned)));
            // ordered on the launch stream before the first sq_attention
            EVK_HIP(hipMemsetAsync(g_sq_cnt, 0, heads * sizeof(unsigned), st));
            g_sq_cnt_n = heads;
        }
    }
    a.part = g_sq_part;
    a.counters = g_sq_cnt;
    const bool one = chunk <= 256 / (dh / 8);  // a split is one pass
    auto launch = [&](auto D) {
        constexpr int DH = decltype(D)::value;
        const dim3 grid(heads, nsplit);
        if (one) hipLaunchKernelGGL((sq_attention<DH, 1>), grid, dim3(256), 0, st, a);
        else hipLaunchKernelGGL((sq_attention<DH, SQ_U>), grid, dim3(256), 0, st, a);
    };
    switch (dh) {
        case 16: launch(std::integral_constant<int, 16>{}); break;
        case 32: launch(std::integral_constant<int, 32>{}); break;
        case 64: launch(std::integral_constant<int, 64>{}); break;
        case 128: launch(std::integral_constant<int, 128>{}); break;
        default: launch(std::integral_constant<int, 256>{}); break;
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? EVKHIP_OK : check_hip(e, "sq_attention launch");
}

int kv_cache_write_launch(const f16* src, f16* cache, int batch, int n, int D, int max_seq, int pos0,
                          hipStream_t st) {
    const int64_t total = (int64_t)batch * n * D;
    if (total == 0) return EVKHIP_OK;
    const int vec = (D % 8 == 0) && aligned16(src) && aligned16(cache);
    const int64_t threads = vec ? total / 8 : total;
    hipLaunchKernelGGL(kv_write_k, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, src, cache, total, n,
                       D, max_seq, pos0, vec);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? EVKHIP_OK : check_hip(e, "kv_cache_write launch");
}

int rms_norm_launch(const f16* in, f16* out, int64_t rows, int D, float eps, hipStream_t st) {
    if (rows == 0) return EVKHIP_OK;
    const dim3 grid((unsigned)((rows + 3) / 4));
    // up to 64 values a lane has one of them either way, without pieces of 8
    // that most lanes do not hold (100000 x 16: 16.0 us, in registers 17.8)
    if (D <= 64 || D % 8 || D > 4096) hipLaunchKernelGGL(rms_norm_k, grid, dim3(256), 0, st, in, out, rows, D, eps);
    else if (D <= 512) hipLaunchKernelGGL(rms_norm_reg_k<1>, grid, dim3(256), 0, st, in, out, rows, D, eps);
    else if (D <= 1024) hipLaunchKernelGGL(rms_norm_reg_k<2>, grid, dim3(256), 0, st, in, out, rows, D, eps);
    else if (D <= 2048) hipLaunchKernelGGL(rms_norm_reg_k<4>, grid, dim3(256), 0, st, in, out, rows, D, eps);
    else hipLaunchKernelGGL(rms_norm_reg_k<8>, grid, dim3(256), 0, st, in, out, rows, D, eps);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? EVKHIP_OK : check_hip(e, "rms_norm launch");
}

int rope_launch(const f16* in, f16* out, int B, int S, int E, float base, int pos0, int hd, hipStream_t st) {
    int64_t n = (int64_t)B * S * (E / 2);
    if (n == 0) return EVKHIP_OK;
    hipLaunchKernelGGL(rope_k, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, in, out, B, S, E, base, pos0,
                       hd);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? EVKHIP_OK : check_hip(e, "rope launch");
}

int gelu_launch(const f16* in, f16* out, int64_t n, hipStream_t st) {
    if (n == 0) return EVKHIP_OK;
    hipLaunchKernelGGL(gelu_k, dim3((unsigned)((n + 2047) / 2048)), dim3(256), 0, st, in, out, n);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? EVKHIP_OK : check_hip(e, "gelu launch");
}

int add_launch(const f16* a, const f16* b, f16* c, int64_t n, hipStream_t st) {
    if (n == 0) return EVKHIP_OK;
    hipLaunchKernelGGL(add_k, dim3((unsigned)((n + 2047) / 2048)), dim3(256), 0, st, a, b, c, n);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? EVKHIP_OK : check_hip(e, "add launch");
}

int embed_launch(const f16* table, const uint16_t* idx, f16* out, int64_t n_idx, int dim, int vocab,
                 hipStream_t st) {
    if (n_idx == 0 || dim == 0) return EVKHIP_OK;
    // 8 values a thread unless a row's last, partial piece would cost more
    // than the others save: short rows of a length off 8, or few of them.  us,
    // one value and 8 a thread: 20000 x 7 1.9 and 3.0, 100000 x 31 5.6 and 6.7,
    // 100 x 255 1.8 and 2.6; 20000 x 65 3.2 and 2.7, 1000 x 1001 2.8 and 2.4.
    const bool by_value = dim % 8 && (dim < 32 || n_idx * dim < (1 << 19));
    const int pieces = by_value ? dim : (dim + 7) / 8;
    const dim3 grid((unsigned)((n_idx * pieces + 255) / 256));
    if (by_value) hipLaunchKernelGGL(embed_k<1>, grid, dim3(256), 0, st, table, idx, out, n_idx, dim, pieces, vocab);
    else hipLaunchKernelGGL(embed_k<8>, grid, dim3(256), 0, st, table, idx, out, n_idx, dim, pieces, vocab);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? EVKHIP_OK : check_hip(e, "embed launch");
}

int greedy_launch(const f16* logits, uint16_t* out, int B, int S, int V, int position, int token_base,
                  int token_count, hipStream_t st) {
    if (B == 0) return EVKHIP_OK;
    auto launch = [&](auto nt, auto w, auto ld) {
        constexpr int NT = decltype(nt)::value, W = decltype(w)::value, LD = decltype(ld)::value;
        hipLaunchKernelGGL((greedy_k<NT, W, LD>), dim3(B), dim3(NT), 0, st, logits, out, S, V, position, token_base,
                           token_count);
    };
    using std::integral_constant;
    // The latency of one row's loads and of the comparisons behind them, or
    // many rows' workgroups.  us for rows of 32, 2000, 8192 and 32000 values,
    // one row: 256 x 1 2.2, 3.4, 7.4, 22.9; 256 x 8 2.7, 2.8, 4.7, 12.7; 512 x
    // 2 x 8 3.2, 3.2, 3.7, 7.6; 1024 x 2 x 8 3.5, 3.6, 4.2, 6.4.  2048 rows:
    // 3.4, 5.1, 11.2, 52; 3.9, 4.9, 9.8, 30; 6.3, 7.0, 10.2, 28; 12, 12, 17, 31.
    constexpr integral_constant<int, 1> one{};
    constexpr integral_constant<int, 2> two{};
    constexpr integral_constant<int, 8> eight{};
    if (token_count <= 512) launch(integral_constant<int, 256>{}, one, one);
    else if (token_count <= 4096) launch(integral_constant<int, 256>{}, eight, one);
    else if (token_count <= 8192 || B > device_cu_count()) launch(integral_constant<int, 512>{}, eight, two);
    else launch(integral_constant<int, 1024>{}, eight, two);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? EVKHIP_OK : check_hip(e, "greedy_sample launch");
}

}  // namespace evkhip
