// attn_prefill.hip -- exact causal attention of a prompt chunk.
//
// The arithmetic is the decode path's (attention.hip: onlineAttentionGroup4F16
// model.go:3527-3588), per query head and token: eight fma chains over the
// elements 8i + j of a dot and the 8 -> 4 -> 2 -> 1 tree, times scale; the
// maximum; fastExpF32; the denominator and every output element summed in
// position order.  Each of these chains is a K loop of a float32 matrix
// product, and v_mfma_f32_16x16x4 evaluates exactly such a chain: four fmas
// in the order k = 0 .. 3, each rounded (subnormals, infinities and zero signs
// included; the probe library's test compares them), so whole 16 x 16 tiles of scores and outputs run on the matrix
// cores with the reference's bits.  Per kv head the query rows of a chunk are
// numbered R = token * kvmul + head; a query tile is 16 of them, so one pass
// over K and V serves 16 rows where a workgroup per (head, token) read them
// once per row.
//
//   scores   wave = (query tile, 128 positions).  D = K q: row m of the
//            16-position tile is position 4 (m % 4) + m / 4, so register r of
//            lane (g, c) is position 4r + g of query row c, which is the A
//            operand of the values product as it stands.  Lane (i, m) of the
//            K operand holds the 16 bytes 8 (4a + i) .. + 7 of its row, and
//            half j of them feeds chain j: K is read row-major, as stored.
//            Positions past a row's own end are -inf.  Scores go to scratch
//            as [kv head][query tile][position tile][lane][4], with the
//            maximum per row and 128 positions.
//   values   workgroup = query tile, HD / 32 waves of 32 elements each and one
//            wave for the denominators.  Steps of 64 positions: the value
//            waves exponentiate the step's weights into LDS (one barrier),
//            then run out = fma(w, v, out) over them.  Column c of output
//            tile dt is element 32 v + 2 c + dt, so a lane reads V by dwords.
//
// A 512-token prompt through two 8B-shaped layers at positions 0 / 3500 went
// from 2433 / 7434 us to 1885 / 2872 us; in a 3000-token prompt the scores and
// values launches take 81 and 153 us on average.  No cycle of an f32 MFMA runs
// under VALU work here (the coexecution counter stays at 0), so the two add up:
// 57 percent of the SIMDs' busy cycles MFMA and 32 VALU in the scores launch, 30
// and 35 in the values launch, whose waves also wait for one another at each
// step's barrier.
#include <algorithm>

#include "attn_exp.h"

namespace gllm {

typedef float f4v __attribute__((ext_vector_type(4)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));

constexpr int kPaChunk = 128;  // positions per scores wave
constexpr int kPaStep = 64;    // positions per values step

struct PaArgs {
    const float* q;        // [p][n_heads][HD]
    const uint16_t *K, *V; // the layer's cache rows from `start` on
    int kv_dim, n_kv, kvmul, p;
    int span0, span_max;   // token t attends span0 + t positions; span_max = span0 + p - 1
    int q_tiles, p_tiles, chunks;
    float scale;
    float* scores;         // [n_kv][q_tiles][p_tiles][64][4]
    float* cmax;           // [n_kv][q_tiles][chunks][16]
    float* out;            // [p][n_heads][HD]
};

// Positions that query row R (of p * kvmul; later rows repeat the last) attends.
__device__ __forceinline__ int pa_span(const PaArgs& a, int R) {
    return a.span0 + min(R, a.p * a.kvmul - 1) / a.kvmul;
}

template <int HD>
__global__ __launch_bounds__(256) void attn_prefill_scores_kernel(PaArgs a) {
    constexpr int NA = HD / 32;  // 16-byte pieces of a K row per lane
    const int kv = blockIdx.x, lane = threadIdx.x & 63;
    const int g = lane >> 4, c = lane & 15;
    const int qt = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t0 = blockIdx.z * kPaChunk;
    if (qt >= a.q_tiles || t0 >= pa_span(a, 16 * qt + 15)) return;  // whole wave
    const int R = min(16 * qt + c, a.p * a.kvmul - 1);
    const int n = pa_span(a, 16 * qt + c);  // this lane's query row
    const float* qr = a.q + ((size_t)(R / a.kvmul) * a.n_kv * a.kvmul + kv * a.kvmul + R % a.kvmul) * HD + 8 * g;
    f4v qf[NA][2];
#pragma unroll
    for (int i = 0; i < NA; i++) {
        qf[i][0] = *(const f4v*)(qr + 32 * i);
        qf[i][1] = *(const f4v*)(qr + 32 * i + 4);
    }
    const uint16_t* Kg = a.K + (size_t)kv * HD + 8 * g;
    const int row = 4 * (c & 3) + (c >> 2);  // this lane's position of a tile
    auto load = [&](int t, h8v (&k)[NA]) __attribute__((always_inline)) {
        const uint16_t* src = Kg + (size_t)min(t + row, a.span_max - 1) * a.kv_dim;
#pragma unroll
        for (int i = 0; i < NA; i++) k[i] = *(const h8v*)(src + 32 * i);
    };
    const int tiles = min(kPaChunk / 16, a.p_tiles - t0 / 16);
    float* dst = a.scores + (((size_t)kv * a.q_tiles + qt) * a.p_tiles + t0 / 16) * 256 + 4 * lane;
    float mx = -__int_as_float(0x7f800000);
    h8v cur[NA], nxt[NA];
    load(t0, cur);
#pragma unroll 1
    for (int it = 0; it < tiles; it++) {
        load(t0 + 16 * (it + 1), nxt);
        f4v y[8];
#pragma unroll
        for (int i = 0; i < NA; i++)
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const f4v z = {0.0f, 0.0f, 0.0f, 0.0f};
                y[j] = __builtin_amdgcn_mfma_f32_16x16x4f32((float)cur[i][j], qf[i][j >> 2][j & 3], i ? y[j] : z, 0, 0, 0);
            }
        f4v s;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float s0 = y[0][r] + y[4][r], s1 = y[1][r] + y[5][r];
            const float s2 = y[2][r] + y[6][r], s3 = y[3][r] + y[7][r];
            const float v = ((s0 + s1) + (s2 + s3)) * a.scale;
            s[r] = t0 + 16 * it + 4 * r + g < n ? v : -__int_as_float(0x7f800000);
            mx = fmaxf(mx, s[r]);
        }
        *(f4v*)(dst + 256 * it) = s;
#pragma unroll
        for (int i = 0; i < NA; i++) cur[i] = nxt[i];
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    if (g == 0) a.cmax[(((size_t)kv * a.q_tiles + qt) * a.chunks + blockIdx.z) * 16 + c] = mx;
}

template <int HD>
__global__ __launch_bounds__(2 * HD + 64) void attn_prefill_values_kernel(PaArgs a) {
    constexpr int NV = HD / 32;   // value waves
    constexpr int NE = 4 / NV;    // position tiles of a step that a value wave exponentiates
    __shared__ __attribute__((aligned(16))) f4v wts[2][kPaStep / 16][64];
    __shared__ float red[16][4 * (NV + 1)], rmax[16], rinv[16];
    const int kv = blockIdx.x, qt = a.q_tiles - 1 - (int)blockIdx.y;  // the longest spans first
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, c = lane & 15;
    const int n_min = pa_span(a, 16 * qt), n_max = pa_span(a, 16 * qt + 15);
    const int steps = (n_max + kPaStep - 1) / kPaStep;
    const bool chain = w < NV;
    const f4v* S = (const f4v*)a.scores + ((size_t)kv * a.q_tiles + qt) * a.p_tiles * 64 + lane;
    const uint16_t* Vg = a.V + (size_t)kv * HD + 32 * w + 2 * c;
    f4v sc[NE], sn[NE];
    uint32_t vc[16], vn[16];  // [tile of the step][r]: the lane's dword of position 16 tile + 4r + g
    auto load_s = [&](int s, f4v (&x)[NE]) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < NE; e++) x[e] = S[(size_t)min(4 * s + NE * w + e, a.p_tiles - 1) * 64];
    };
    auto load_v = [&](int s, uint32_t (&x)[16]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 16; i++)
            x[i] = *(const uint32_t*)(Vg + (size_t)min(kPaStep * s + 4 * i + g, a.span_max - 1) * a.kv_dim);
    };
    if (chain) {
        load_s(0, sc);
        load_v(0, vc);
    }
    {   // the rows' maxima from the scores launch's
        const float* cm = a.cmax + ((size_t)kv * a.q_tiles + qt) * a.chunks * 16;
        const int nch = (n_max + kPaChunk - 1) / kPaChunk;
        float m = -__int_as_float(0x7f800000);
        for (int i = tid >> 4; i < nch; i += 4 * (NV + 1)) m = fmaxf(m, cm[16 * i + c]);
        red[c][tid >> 4] = m;
        __syncthreads();
        if (tid < 16) {
            for (int i = 1; i < 4 * (NV + 1); i++) m = fmaxf(m, red[tid][i]);
            rmax[tid] = m;
        }
        __syncthreads();
    }
    const float mx = rmax[c];
    f4v acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
    float denom = 0.0f;
#pragma unroll 1
    for (int s = 0; s < steps; s++) {
        f4v (*W)[64] = wts[s & 1];
        if (chain) {
            // the next step's loads first; tiles past the span hold no scores,
            // so their weights are set, not computed from what is there
            load_s(s + 1, sn);
            load_v(s + 1, vn);
#pragma unroll
            for (int e = 0; e < NE; e++) {
                float x[4], y[4];
#pragma unroll
                for (int r = 0; r < 4; r++) x[r] = sc[e][r] - mx;
                fast_exp_n(x, y);
                const bool in = kPaStep * s + 16 * (NE * w + e) < n_max;
                W[NE * w + e][lane] = in ? f4v{y[0], y[1], y[2], y[3]} : f4v{0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
        wait_lgkm0();
        lds_barrier();
        if (chain) {
#pragma unroll
            for (int tl = 0; tl < 4; tl++) {
                const int t = kPaStep * s + 16 * tl;
                if (t >= n_max) break;  // uniform
                const f4v wv = W[tl][lane];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const h2v v2 = __builtin_bit_cast(h2v, vc[4 * tl + r]);
                    const float v0 = (float)v2[0], v1 = (float)v2[1];
                    if (t + 4 * r + 3 < n_min) {
                        acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[r], v0, acc[0], 0, 0, 0);
                        acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[r], v1, acc[1], 0, 0, 0);
                        continue;
                    }
                    // the ends of the tile's tokens: a position past a row's
                    // end has weight 0, which adds nothing unless its v is
                    // not finite
                    const bool odd = !(fabsf(v0) <= 65504.0f) || !(fabsf(v1) <= 65504.0f);
                    if (__ballot(odd) == 0) {
                        acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[r], v0, acc[0], 0, 0, 0);
                        acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[r], v1, acc[1], 0, 0, 0);
                        continue;
                    }
                    // one position at a time, kept only by the rows that reach it
                    for (int k = 0; k < 4; k++) {
                        const bool on = g == k;
                        const f4v d0 = __builtin_amdgcn_mfma_f32_16x16x4f32(on ? wv[r] : 0.0f, on ? v0 : 0.0f, acc[0], 0, 0, 0);
                        const f4v d1 = __builtin_amdgcn_mfma_f32_16x16x4f32(on ? wv[r] : 0.0f, on ? v1 : 0.0f, acc[1], 0, 0, 0);
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const bool keep = t + 4 * r + k < pa_span(a, 16 * qt + 4 * g + i);
                            acc[0][i] = keep ? d0[i] : acc[0][i];
                            acc[1][i] = keep ? d1[i] : acc[1][i];
                        }
                    }
                }
            }
#pragma unroll
            for (int e = 0; e < NE; e++) sc[e] = sn[e];
#pragma unroll
            for (int i = 0; i < 16; i++) vc[i] = vn[i];
        } else {
            // position order: 4r + g (weights past a row's end are 0)
#pragma unroll
            for (int tl = 0; tl < 4; tl++) {
                f4v x[4];
#pragma unroll
                for (int k = 0; k < 4; k++) x[k] = W[tl][16 * k + c];
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int k = 0; k < 4; k++) denom = denom + x[k][r];
            }
        }
    }
    if (!chain && lane < 16) rinv[lane] = denom > 0.0f ? 1.0f / denom : 1.0f;
    __syncthreads();
    if (!chain) return;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int R = 16 * qt + 4 * g + i;
        if (R >= a.p * a.kvmul) continue;
        const float inv = rinv[4 * g + i];
        float* o = a.out + ((size_t)(R / a.kvmul) * a.n_kv * a.kvmul + kv * a.kvmul + R % a.kvmul) * HD + 32 * w + 2 * c;
        *(float2*)o = make_float2(acc[0][i] * inv, acc[1][i] * inv);
    }
}

// Device floats of scratch that a chunk of p tokens over up to span_max
// positions takes.
size_t attend_prefill_floats(int p, int n_heads, int n_kv, int span_max) {
    const size_t qt = ((size_t)p * (n_heads / n_kv) + 15) / 16;
    return n_kv * qt * ((size_t)(span_max + 15) / 16 * 256 + (size_t)(span_max + kPaChunk - 1) / kPaChunk * 16);
}

// The matrix-core path applies: head_dim 64 or 128 with 16-byte aligned rows.
bool attend_prefill_fits(int hd, int kv_dim_k, int kv_dim_v) {
    return (hd == 64 || hd == 128) && kv_dim_k == kv_dim_v && kv_dim_k % 8 == 0;
}

// Exact attention of p consecutive tokens: token t attends the span0 + t
// positions from the rows K / V on.  scratch: attend_prefill_floats floats.
int attend_prefill(const float* d_q, const uint16_t* K, const uint16_t* V, int kv_dim, int n_heads, int n_kv, int hd,
                   int span0, int p, float scale, float* scratch, float* d_out, hipStream_t s) {
    PaArgs a{};
    a.q = d_q;
    a.K = K;
    a.V = V;
    a.kv_dim = kv_dim;
    a.n_kv = n_kv;
    a.kvmul = n_heads / n_kv;
    a.p = p;
    a.span0 = span0;
    a.span_max = span0 + p - 1;
    a.q_tiles = (p * a.kvmul + 15) / 16;
    a.p_tiles = (a.span_max + 15) / 16;
    a.chunks = (a.span_max + kPaChunk - 1) / kPaChunk;
    a.scale = scale;
    a.scores = scratch;
    a.cmax = scratch + (size_t)n_kv * a.q_tiles * a.p_tiles * 256;
    a.out = d_out;
    const dim3 gs(n_kv, (a.q_tiles + 3) / 4, a.chunks), gv(n_kv, a.q_tiles);
    if (hd == 128) {
        hipLaunchKernelGGL(attn_prefill_scores_kernel<128>, gs, dim3(256), 0, s, a);
        GLLM_HIP(hipGetLastError());
        hipLaunchKernelGGL(attn_prefill_values_kernel<128>, gv, dim3(320), 0, s, a);
    } else {
        hipLaunchKernelGGL(attn_prefill_scores_kernel<64>, gs, dim3(256), 0, s, a);
        GLLM_HIP(hipGetLastError());
        hipLaunchKernelGGL(attn_prefill_values_kernel<64>, gv, dim3(192), 0, s, a);
    }
    GLLM_HIP(hipGetLastError());
    return GLLM_OK;
}

}  // namespace gllm
