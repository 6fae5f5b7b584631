// prefill.hip -- batched products on the matrix cores: Q4_K, Q5_K, Q6_K, Q8_0
// and Q4_0 x Q8_K.  Q4_K's arithmetic first; the others' stands at their kernels.
//
// matvecBatchQ8 (kernels_amd64.go:470-581) runs the batch-1 row kernel
// q4kDotQ8KRow (kernels_amd64.s:437-543) once per (row, token), so a batched
// result must equal the per-token one bit for bit.  That kernel keeps eight
// AVX2 lanes per row; lane k owns the 32 elements {32j + 4k + i : j < 8,
// i < 4} of every 256-element block b and runs two float chains over b:
//   accF[k] = fma(float(I_bk), d_b * xscale_b, accF[k])
//   accM[k] = fma(dmin_b, float(m_bk) * xsum_bk, accM[k])
// with the exact integer I_bk = sum over its 32 elements of sc_j * q4 * q8,
// and ends with tree8(accF - accM).
//
// Here I_bk comes from v_mfma_f32_16x16x32_f16: the A operand holds
// sc_j * q4 (<= 63 * 15 = 945, exact in f16), the B operand q8 (exact in
// f16), and every partial sum of 32 products stays below 2^24, so the fp32
// accumulation is exact in any order and equals the int32 lane sum.  The
// float chains then run per (row, token, lane) in VALU registers in the
// reference's order.
//
// K order: lane k's elements are numbered kappa = 4j + i, which is the order
// of the lane-permuted Q8K activations (q8perm_offset) and, for the weights,
// of the upload repack: lane k's 16 nibble bytes sit at 16 + 16k, byte
// 4s + i holding elements kappa = 8s + i (low nibble, sub-block 2s) and
// 8s + 4 + i (high nibble, sub-block 2s + 1).  MFMA lane L supplies
// kappa = 8(L/16) .. 8(L/16) + 7 of both operands, i.e. one weight dword.
//
// Three kinds of kernel follow: prefill_q4k_mfma_kernel (8 to 16 tokens, where
// the rows fill the GPU or the activations carry no records), the *_lanes_kernels
// (more than 16 tokens, every format below on its own chains) and
// small_lanes_kernel (2 to 16 tokens).  The last two take the activations as
// the A operand and the weights as B.
//
// prefill_q4k_mfma_kernel: a workgroup is four waves over 64 weight rows x 16
// tokens; wave w owns the 16x16 tile of rows 16 w .. + 15.  Per block the
// workgroup stages the tokens' q8 (as f16), xsums and xscales and the rows'
// decoded scales/mins and nibble bytes in LDS (double-buffered, loaded one
// block ahead).  It wins over small_lanes_kernel with many rows, see
// small_batch_fits for both sides.
#include "gllm_common.h"

namespace gllm {

typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

constexpr int kPfBStride = 528;  // bytes per token row of the f16 q8 tile: 512 + 16 (no bank conflicts)
constexpr int kPfWStride = 36;   // dwords per row of the staged weight nibbles: 32 + 4

constexpr int kPfRows = 64, kPfTok = 16, kPfThreads = 256;  // of a workgroup

// One block's staged operands of a workgroup.
struct PfStage {
    uint8_t b16[kPfTok * kPfBStride];
    float xsum[8][kPfTok];        // [lane k][token]
    float xsc[kPfTok];
    uint32_t sch[8][kPfRows];     // [sub-block j][row] half2(sc_j, sc_j)
    uint32_t scn[8][kPfRows];     // [sub-block j][row] half2(-1024 sc_j, -1024 sc_j)
    float m[8][kPfRows];          // [lane k][row]
    float d[kPfRows];
    float dmin[kPfRows];
    // nibble dwords per row as [group s][lane k] (lane (g, c) of a wave reads
    // its 8 dwords as 32 contiguous bytes); 36-dword rows keep the 16 rows'
    // 16-byte reads on distinct banks
    uint32_t wa[kPfRows][kPfWStride];
};

// four signed bytes -> two half2 words holding the same integers
__device__ __forceinline__ void i8x4_to_h(uint32_t w, uint32_t& lo, uint32_t& hi) {
    const uint32_t u = w ^ 0x80808080u;  // c + 128, as unsigned bytes
    const uint32_t a = __builtin_amdgcn_perm(0x64646464u, u, 0x05010400u);  // 1024 + u0, 1024 + u1
    const uint32_t b = __builtin_amdgcn_perm(0x64646464u, u, 0x05030402u);  // 1024 + u2, 1024 + u3
    typedef _Float16 h2v __attribute__((ext_vector_type(2)));
    const h2v bias = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    h2v ha = __builtin_bit_cast(h2v, a) + bias;  // exact: integers below 2048
    h2v hb = __builtin_bit_cast(h2v, b) + bias;
    lo = __builtin_bit_cast(uint32_t, ha);
    hi = __builtin_bit_cast(uint32_t, hb);
}

// one weight dword (4 nibble bytes of one lane and sub-block pair) -> the
// 8 f16 A values sc_lo * low nibbles, sc_hi * high nibbles
__device__ __forceinline__ h8v dequant_a(uint32_t w, uint32_t sch_lo, uint32_t scn_lo,
                                         uint32_t sch_hi, uint32_t scn_hi) {
    typedef _Float16 h2v __attribute__((ext_vector_type(2)));
    const uint32_t lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu;
    const h2v p0 = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, lo, 0x05010400u));
    const h2v p1 = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, lo, 0x05030402u));
    const h2v p2 = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, hi, 0x05010400u));
    const h2v p3 = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, hi, 0x05030402u));
    const h2v sl = __builtin_bit_cast(h2v, sch_lo), nl = __builtin_bit_cast(h2v, scn_lo);
    const h2v sh = __builtin_bit_cast(h2v, sch_hi), nh = __builtin_bit_cast(h2v, scn_hi);
    // (1024 + q) * sc - 1024 * sc == q * sc exactly: one rounding of an exact
    // value below 2048
    const h2v a0 = __builtin_elementwise_fma(p0, sl, nl);
    const h2v a1 = __builtin_elementwise_fma(p1, sl, nl);
    const h2v a2 = __builtin_elementwise_fma(p2, sh, nh);
    const h2v a3 = __builtin_elementwise_fma(p3, sh, nh);
    h8v r;
    r[0] = a0[0]; r[1] = a0[1]; r[2] = a1[0]; r[3] = a1[1];
    r[4] = a2[0]; r[5] = a2[1]; r[6] = a3[0]; r[7] = a3[1];
    return r;
}

struct PfArgs {
    const uint8_t* w;  // repacked Q4_K rows
    size_t rb;         // bytes per row
    int rows, blocks;
    ActQ8 act;         // p tokens of Q8K activations
    int p;
    float* out;        // out[t * out_stride + r]
    int out_stride;
};

// Staging registers of one block, mapped so that every LDS store of a wave hits
// distinct banks:
//   q8: thread = (token tid / 16, part tid % 16): q8 bytes 8 part .. + 7 and
//       128 + 8 part .. + 7, written as f16 at 16 part and 256 + 16 part of the
//       token's row;
//   threads 0 .. 2 kPfTok - 1 one xsum quad, threads 0 .. kPfTok - 1 one xscale;
//   unit u = (sub-block j = u / kPfRows, row u % kPfRows), units tid and tid +
//   kPfThreads: the row's block header and the 16 nibble bytes of lane k = j.
struct PfRegs {
    static constexpr int NH = 8 * kPfRows / kPfThreads;  // header units per thread
    uint32_t q[4];
    f4v xs;
    float xc;
    u4v h[NH];
    u4v w[NH];
};

__device__ __forceinline__ void pf_load(const PfArgs& a, int row0, int tok0, int b,
                                        PfRegs& r) {
    const int tid = threadIdx.x;
    const int cols = a.blocks * 256;
    {
        const int t = min(tok0 + (tid >> 4), a.p - 1);
        const int8_t* src = a.act.q8perm + (size_t)t * cols + (size_t)b * 256 + 8 * (tid & 15);
        const uint2 lo = *(const uint2*)src, hi = *(const uint2*)(src + 128);
        r.q[0] = lo.x; r.q[1] = lo.y; r.q[2] = hi.x; r.q[3] = hi.y;
    }
    if (tid < 2 * kPfTok) {
        const int t = min(tok0 + (tid >> 1), a.p - 1);
        r.xs = *(const f4v*)(a.act.xs32 + (size_t)t * (cols / 32) + b * 8 + 4 * (tid & 1));
    }
    if (tid < kPfTok) r.xc = a.act.xscale[(size_t)min(tok0 + tid, a.p - 1) * a.blocks + b];
#pragma unroll
    for (int i = 0; i < PfRegs::NH; i++) {
        const int u = tid + kPfThreads * i;
        const int row = min(row0 + u % kPfRows, a.rows - 1);
        const uint8_t* rp = a.w + (size_t)row * a.rb;
        r.h[i] = *(const u4v*)(rp + q4k_hdr_off(b));
        r.w[i] = *(const u4v*)(rp + q4k_nib_off(a.blocks, b) + 16 * (u / kPfRows));
    }
}

__device__ __forceinline__ void pf_store(const PfRegs& r, PfStage& st) {
    const int tid = threadIdx.x;
    {
        uint32_t v[8];
        i8x4_to_h(r.q[0], v[0], v[1]);
        i8x4_to_h(r.q[1], v[2], v[3]);
        i8x4_to_h(r.q[2], v[4], v[5]);
        i8x4_to_h(r.q[3], v[6], v[7]);
        uint8_t* row = st.b16 + (tid >> 4) * kPfBStride + 16 * (tid & 15);
        *(u4v*)row = u4v{v[0], v[1], v[2], v[3]};
        *(u4v*)(row + 256) = u4v{v[4], v[5], v[6], v[7]};
    }
    if (tid < 2 * kPfTok) {
        const int t = tid >> 1, k0 = 4 * (tid & 1);
        st.xsum[k0][t] = r.xs.x;
        st.xsum[k0 + 1][t] = r.xs.y;
        st.xsum[k0 + 2][t] = r.xs.z;
        st.xsum[k0 + 3][t] = r.xs.w;
    }
    if (tid < kPfTok) st.xsc[tid] = r.xc;
#pragma unroll
    for (int i = 0; i < PfRegs::NH; i++) {
        // getScaleMinK4 (simd.go:1672-1677) for sub-block j
        const int u = tid + kPfThreads * i;
        const int row = u % kPfRows, j = u / kPfRows;
        const uint32_t s03 = r.h[i].y, s47 = r.h[i].z, s811 = r.h[i].w;
        uint32_t sc, mn;
        if (j < 4) {
            sc = (s03 >> (8 * j)) & 63u;
            mn = (s47 >> (8 * j)) & 63u;
        } else {
            const int jj = j - 4;
            const uint32_t b8 = (s811 >> (8 * jj)) & 0xffu;
            sc = (b8 & 15u) | (((s03 >> (8 * jj + 6)) & 3u) << 4);
            mn = (b8 >> 4) | (((s47 >> (8 * jj + 6)) & 3u) << 4);
        }
        const _Float16 hs = (_Float16)(float)sc, hn = (_Float16)(-1024.0f * (float)sc);
        const uint32_t bs = __builtin_bit_cast(uint16_t, hs), bn = __builtin_bit_cast(uint16_t, hn);
        st.sch[j][row] = bs | (bs << 16);
        st.scn[j][row] = bn | (bn << 16);
        st.m[j][row] = (float)mn;
        if (j == 0) {
            st.d[row] = f16_bits_to_f32(r.h[i].x & 0xffffu);
            st.dmin[row] = f16_bits_to_f32(r.h[i].x >> 16);
        }
        // lane k = j's dwords for groups s = 0..3
        st.wa[row][0 * 8 + j] = r.w[i].x;
        st.wa[row][1 * 8 + j] = r.w[i].y;
        st.wa[row][2 * 8 + j] = r.w[i].z;
        st.wa[row][3 * 8 + j] = r.w[i].w;
    }
}

__global__ __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_q4k_mfma_kernel(PfArgs a) {
    __shared__ __align__(16) PfStage stage[2];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane >> 4, c = lane & 15;
    const int row0 = blockIdx.x * kPfRows, tok0 = blockIdx.y * kPfTok;
    // D layout: rows 4g + i of the wave's 16, token c
    const int lr = 16 * wave + 4 * g;

    float accF[4][8], accM[4][8];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int k = 0; k < 8; k++) accF[i][k] = accM[i][k] = 0.0f;

    // one block's products from a staged LDS tile
    auto block = [&](const PfStage& st) __attribute__((always_inline)) {
        // this lane's A row (MFMA row c of the wave's 16): its 8 nibble dwords
        const u4v wq0 = *(const u4v*)&st.wa[16 * wave + c][8 * g];
        const u4v wq1 = *(const u4v*)&st.wa[16 * wave + c][8 * g + 4];
        const uint32_t wq[8] = {wq0.x, wq0.y, wq0.z, wq0.w, wq1.x, wq1.y, wq1.z, wq1.w};
        const uint32_t sh_lo = st.sch[2 * g][16 * wave + c], sn_lo = st.scn[2 * g][16 * wave + c];
        const uint32_t sh_hi = st.sch[2 * g + 1][16 * wave + c], sn_hi = st.scn[2 * g + 1][16 * wave + c];
        // F chain factors d * xscale per D row
        const f4v dv = *(const f4v*)&st.d[lr];
        const f4v dm = *(const f4v*)&st.dmin[lr];
        const float xc = st.xsc[c];
        float dxs[4];
#pragma unroll
        for (int i = 0; i < 4; i++) dxs[i] = dv[i] * xc;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const h8v av = dequant_a(wq[k], sh_lo, sn_lo, sh_hi, sn_hi);
            const h8v bv = *(const h8v*)(st.b16 + c * kPfBStride + 64 * k + 16 * g);
            const f4v z = {0.0f, 0.0f, 0.0f, 0.0f};
            const f4v dI = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bv, z, 0, 0, 0);
            // M chain operands: mins of the lane's 4 D rows, xsum of its token
            const f4v mk = *(const f4v*)&st.m[k][lr];
            const float xk = st.xsum[k][c];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                accF[i][k] = fmaf(dI[i], dxs[i], accF[i][k]);
                const float mx = mk[i] * xk;
                accM[i][k] = fmaf(dm[i], mx, accM[i][k]);
            }
        }
    };

    // Two staging register sets: the global loads of block b + 2 are issued
    // while block b is computed and land in LDS after block b + 1 is.  The
    // loads are unconditional (past the end they re-read the last block):
    // under a branch the compiler's vmcnt wait for the older set would also
    // wait for the newer one and cancel the prefetch.
    const int nb = a.blocks;
    PfRegs r0, r1;
    pf_load(a, row0, tok0, 0, r0);
    pf_store(r0, stage[0]);
    pf_load(a, row0, tok0, min(1, nb - 1), r1);
    __syncthreads();
#pragma unroll 1
    for (int b = 0; b < nb; b += 2) {
        pf_load(a, row0, tok0, min(b + 2, nb - 1), r0);
        block(stage[0]);
        if (b + 1 < nb) pf_store(r1, stage[1]);
        __syncthreads();
        if (b + 1 >= nb) break;
        pf_load(a, row0, tok0, min(b + 3, nb - 1), r1);
        block(stage[1]);
        if (b + 2 < nb) pf_store(r0, stage[0]);
        __syncthreads();
    }
    // tree8 of the reference's horizontal sum, then the (row, token) store
    const int t = tok0 + c;
    if (t < a.p) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = row0 + lr + i;
            if (r >= a.rows) continue;
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] = accF[i][k] - accM[i][k];
            const float s0 = v[0] + v[4], s1 = v[1] + v[5], s2 = v[2] + v[6], s3 = v[3] + v[7];
            a.out[(size_t)t * a.out_stride + r] = (s0 + s1) + (s2 + s3);
        }
    }
}

static void launch_pf(const PfArgs& a, hipStream_t s) {
    dim3 grid((a.rows + kPfRows - 1) / kPfRows, (a.p + kPfTok - 1) / kPfTok);
    hipLaunchKernelGGL(prefill_q4k_mfma_kernel, grid, dim3(kPfThreads), 0, s, a);
}

// --- more than 16 activation rows: one pair of AVX2 lanes per wave ---------
// A workgroup of sixteen waves covers 64 weight rows x 64 tokens.  The eight
// AVX2 lanes k of a row never meet before the final tree, so the waves split
// by lane: wave (rq, kp) = (w >> 2, w & 3) owns rows 16 rq .. + 15, all 64
// tokens and the lanes kp and kp + 4, the first pair the tree adds.  A weight
// nibble then belongs to one wave: it is dequantised once, in that wave's
// registers, straight into the MFMA operand, with no f16 copy of the weights
// in LDS, and 64 accumulator registers leave room for four waves per SIMD.
// The products take the activations as the A operand and the weights as B,
// so D has token 16 tt + 4g + i in register i and weight row 16 rq + c in
// lane (g, c): a row's factors are one register per lane, and the stores run
// along the rows.  The two outer products of a block, m * xsum and
// d * xscale, come from v_mfma_f32_16x16x1 with K = 1: one exact float32
// product per output, rounded once, as the VALU's (a zero product may lose
// its sign, which a chain that starts at +0 does not show).  Four 16-token
// tiles are its four blocks, so an operand is one register and one dword of
// LDS per lane.  Left to the VALU are the two chain steps per output:
//   accF = fma(I, d * xscale, accF); accM = fma(dmin, m * xsum, accM).
// Per block the workgroup stages the token tiles' B16 operands, xsums and
// xscales in LDS one block ahead, and each wave its own nibbles and headers
// two blocks ahead (they come from HBM), all by direct copies; one barrier
// per block.  The block loop is unrolled by two, so every LDS address is a
// lane constant plus an immediate.
// Measured at 14336 x 4096 x 512 (with the 9.5 us quantiser launch): 261 us
// for the kernel before it, which staged the dequantised f16 weights in LDS
// and ran all eight lanes of a 16 x 32 tile in a wave (two waves per SIMD,
// LDS traffic 370 KB per block), 195 us with eight waves of 32 rows x 64
// tokens (two per SIMD), 202 us with eight waves of 16 rows x 128 tokens, 175
// us like this.  What is left is issue: per wave and block 128 VALU instructions,
// 64 of them chain steps, and 11 matrix instructions of 16 (f16) and 32 cycles
// (f32); by the counters the SIMDs' busy cycles are 61 percent VALU and 26
// percent MFMA, a quarter of the latter under VALU work.
// Up to kHalfTok tokens the products and chains run on two of the four token
// tiles only (NT = 2).  17 tokens, four / two tiles: 4096 x 14336 Q4_K 78 / 64 us,
// Q5_K 91 / 77, Q6_K 120 / 96, Q8_0 138 / 86.  As a branch inside one kernel it
// also served the last tile of a longer prompt, which gained nothing there
// and cost Q8_0 and Q4_K up to 2 percent at full tiles.
constexpr int kTlRows = 64, kTlTok = 64, kHalfTok = 32;

// Q5_K (q5kDotQ8KRow, kernels_amd64.s:578-663) has the same chains; its codes
// take a fifth bit from the qh plane (sc * code <= 63 * 31, exact in f16), so
// a nibble dword's pairs get one more masked term each: 206 us at 14336 x 4096 x
// 512, where the row kernels, eight tokens at a time, took 2889 us.
template <bool Q5>
struct LnStage {
    uint8_t b16[4 * 8 * 4 * 256];  // [token tile][lane k][group g][token c][8 halves]
    float xsum[4][8][16];          // [token tile][lane k][token c]
    float xs[kTlTok];
    // [wave]: nibbles [lane kp, kp + 4][row c], headers [row c], and for Q5_K
    // the 16 bytes with the two lanes' qh dwords [lane kp, kp + 4][row c]
    uint8_t raw[16][Q5 ? 80 : 48][16];
};

// Direct global -> LDS copies addressed by a wave-uniform base and a 32-bit
// per-lane byte offset (the saddr form), so a copy costs one VGPR.  The s_nop
// is the wait state between the M0 write and the load, as in lds_copy16.
__device__ __forceinline__ void lds_copy16_s(const void* sbase, uint32_t voff, uint32_t lds_dst) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(voff), "s"(sbase), "s"(lds_dst)
                 : "memory", "m0");
}
__device__ __forceinline__ void lds_copy4_s(const void* sbase, uint32_t voff, uint32_t lds_dst) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                 :
                 : "v"(voff), "s"(sbase), "s"(lds_dst)
                 : "memory", "m0");
}

// Workgroup -> tile map.  Workgroup i runs on XCD i % 8 (round robin); the
// eight XCDs form an h x v grid, XCD x taking token-tile group x % h and
// row-tile group x / h, so each XCD reads its share of the weights once and
// its (at most four 64-token tiles' worth of) activations stay in its L2
// while the weight rows stream past.  Within an XCD the token tiles of one
// row tile are consecutive, so they read its weights at about the same time.
struct TlMap {
    int row_tiles, tok_tiles;  // whole problem
    int h, v;                  // XCD grid: h token groups x v row groups
    int tg_size, rg_size;      // token / row tiles per group
};

static TlMap tl_map(int rows, int p) {
    TlMap m;
    m.row_tiles = (rows + kTlRows - 1) / kTlRows;
    m.tok_tiles = (p + kTlTok - 1) / kTlTok;
    m.h = 1;
    while (m.h < 8 && (m.tok_tiles + m.h - 1) / m.h > 4) m.h *= 2;
    m.v = 8 / m.h;
    m.tg_size = (m.tok_tiles + m.h - 1) / m.h;
    m.rg_size = (m.row_tiles + m.v - 1) / m.v;
    return m;
}

typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef float f16v __attribute__((ext_vector_type(16)));

// One nibble dword as eight f16 values sc_lo * low, sc_hi * high in the
// element order of B16 (bytes 0, 2, 1, 3).  A masked nibble pair under f16
// exponent bits is 1024 + q (bits 0-3) or 1024 + 16 q (bits 4-7), so with
// s = {sc_lo, sc_hi / 16} and n = -1024 s the fma is exact.
struct NibMasks {  // held in registers: a v_and_or_b32 takes no two literals
    uint32_t lo, hi, exp;
};
__device__ __forceinline__ NibMasks nib_masks() {
    NibMasks m{0x000f000fu, 0x00f000f0u, 0x64006400u};
    asm("" : "+s"(m.lo), "+s"(m.hi), "+v"(m.exp));
    return m;
}
__device__ __forceinline__ h8v dequant_nib(uint32_t w, h2v s, h2v n, const NibMasks& m) {
    const uint32_t v = w >> 8;
    const h2v p0 = __builtin_bit_cast(h2v, (w & m.lo) | m.exp), p1 = __builtin_bit_cast(h2v, (v & m.lo) | m.exp);
    const h2v p2 = __builtin_bit_cast(h2v, (w & m.hi) | m.exp), p3 = __builtin_bit_cast(h2v, (v & m.hi) | m.exp);
    const h2v sl = {s[0], s[0]}, nl = {n[0], n[0]}, sh = {s[1], s[1]}, nh = {n[1], n[1]};
    const h2v a0 = __builtin_elementwise_fma(p0, sl, nl), a1 = __builtin_elementwise_fma(p1, sl, nl);
    const h2v a2 = __builtin_elementwise_fma(p2, sh, nh), a3 = __builtin_elementwise_fma(p3, sh, nh);
    return h8v{a0[0], a0[1], a1[0], a1[1], a2[0], a2[1], a3[0], a3[1]};
}

// The same for Q5_K: bits 0 and 1 of every byte of qh are the fifth bits of
// the low and the high nibbles, at mantissa bits 4 and 8 of their pairs.
__device__ __forceinline__ h8v dequant_q5(uint32_t w, uint32_t qh, h2v s, h2v n, const NibMasks& m) {
    const uint32_t v = w >> 8;
    const uint32_t b0 = m.exp | ((qh << 4) & 0x00100010u), b1 = m.exp | ((qh >> 4) & 0x00100010u);
    const uint32_t b2 = m.exp | ((qh << 7) & 0x01000100u), b3 = m.exp | ((qh >> 1) & 0x01000100u);
    const h2v p0 = __builtin_bit_cast(h2v, (w & m.lo) | b0), p1 = __builtin_bit_cast(h2v, (v & m.lo) | b1);
    const h2v p2 = __builtin_bit_cast(h2v, (w & m.hi) | b2), p3 = __builtin_bit_cast(h2v, (v & m.hi) | b3);
    const h2v sl = {s[0], s[0]}, nl = {n[0], n[0]}, sh = {s[1], s[1]}, nh = {n[1], n[1]};
    const h2v a0 = __builtin_elementwise_fma(p0, sl, nl), a1 = __builtin_elementwise_fma(p1, sl, nl);
    const h2v a2 = __builtin_elementwise_fma(p2, sh, nh), a3 = __builtin_elementwise_fma(p3, sh, nh);
    return h8v{a0[0], a0[1], a1[0], a1[1], a2[0], a2[1], a3[0], a3[1]};
}

// An f16 factor of many chain steps, converted once.  Left alone the compiler
// folds the conversion into each fma as v_fma_mix_f32, which issues more
// slowly (14336 x 4096 x 512 with / without: Q8_0 348 / 305 us, Q4_K 180 /
// 175 us; Q6_K 4096 x 14336 x 333 259 / 245 us).
__device__ __forceinline__ float factor_f16(uint32_t h) {
    float v = f16_bits_to_f32(h & 0xffffu);
    asm("" : "+v"(v));
    return v;
}

// A chain step ends here: the compiler may not sink it past this point.
__device__ __forceinline__ void pin4(float (&v)[4]) {
    asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
}

// (s0 + s1) + (s2 + s3) of the four waves of row group rq, from the exchange
// ex[rq][kp][token tile][i][lane]: wave (rq, kp) stores token tile kp, with
// its offset chains added where a format has them.
template <bool OFF = false>
__device__ __forceinline__ void lanes_store(const PfArgs& a, const float* ex, int row0, int tok0, int rq, int kp,
                                            int lane, f4v off = {}) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; q++) v[q] = ex[(((rq * 4 + q) * 4 + kp) * 4 + i) * 64 + lane];
        const int t = tok0 + 16 * kp + 4 * (lane >> 4) + i, rr = row0 + 16 * rq + (lane & 15);
        float r = (v[0] + v[1]) + (v[2] + v[3]);
        if constexpr (OFF) r = r + off[i];
        if (t < a.p && rr < a.rows) a.out[(size_t)t * a.out_stride + rr] = r;
    }
}

template <bool Q5, int NT>
__global__ __launch_bounds__(1024) void prefill_q4k_lanes_kernel(PfArgs a, TlMap mp) {
    extern __shared__ __attribute__((aligned(16))) uint8_t dyn[];
    LnStage<Q5>* const st = (LnStage<Q5>*)dyn;
    const int id = blockIdx.x, xcd = id & 7, local = id >> 3;
    const int lt = local % mp.tg_size, lrow = local / mp.tg_size;
    const int ttile = (xcd % mp.h) * mp.tg_size + lt, rtile = (xcd / mp.h) * mp.rg_size + lrow;
    if (lrow >= mp.rg_size || ttile >= mp.tok_tiles || rtile >= mp.row_tiles) return;  // whole workgroup
    const int row0 = rtile * kTlRows, tok0 = ttile * kTlTok, tile0 = tok0 / 16;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, c = lane & 15;
    const int kp = w & 3, rq = w >> 2;
    const int nb = a.blocks;

    // Copies of one block's tokens: two 1 KB pieces of B16 (wave w: tile w / 4,
    // lanes k 2 (w % 4), + 1), the tiles' xsums (waves 0, 1) and xscales
    // (wave 2).  Past the end they stay on the last block, so that the counts
    // of copies in flight are constants.
    const int last = a.act.tiles - 1;
    const size_t bstep = (size_t)a.act.tiles * 8192;
    const uint8_t* bsrc = (const uint8_t*)a.act.b16t + (size_t)min(tile0 + rq, last) * 8192 + 2048 * kp;
    const uint32_t xoff = w < 2 ? (uint32_t)(min(tile0 + 2 * w + (lane >> 5), last) * 512 + 16 * (lane & 31))
                                : (uint32_t)min(tok0 + lane, a.p - 1) * nb * 4;
    auto copy_tokens = [&](int b, LnStage<Q5>& S) __attribute__((always_inline)) {
        b = min(b, nb - 1);
        const uint8_t* src = bsrc + b * bstep;
        const uint32_t dst = lds_addr(S.b16 + rq * 8192 + 2048 * kp);
        lds_copy16_s(src, 16 * lane, dst);
        lds_copy16_s(src + 1024, 16 * lane, dst + 1024);
        if (w < 2) lds_copy16_s(a.act.xs32t + (size_t)b * a.act.tiles * 128, xoff, lds_addr(&S.xsum[2 * w][0][0]));
        else if (w == 2) lds_copy4_s(a.act.xscale + b, xoff, lds_addr(&S.xs[0]));
    };
    // The wave's nibbles, lane k = kp + 4 kc of row 16 rq + c in lanes 0-31
    // (kc = 0, 1), and headers, row c in lanes 32-47, of one block after the
    // other (roff: this lane's source offset of the next one)
    const int kc = min(lane >> 4, 2);
    uint32_t roff = (uint32_t)min(row0 + 16 * rq + c, a.rows - 1) * (uint32_t)a.rb +
                    (kc < 2 ? (Q5 ? 16 : 16 * nb) + 16 * (kp + 4 * kc) : 0);
    const uint32_t rstep = Q5 ? 176 : kc < 2 ? 128 : 16;
    constexpr int kRawCopies = Q5 ? 2 : 1;
    auto copy_raw = [&](int b, LnStage<Q5>& S) __attribute__((always_inline)) {
        if (lane < 48) lds_copy16_s(a.w, roff, lds_addr(&S.raw[w][0][0]));
        if constexpr (Q5) {  // the same lanes 0-31: row and lane k, less the lane's nibble offset
            if (lane < 32)
                lds_copy16_s(a.w, roff - (16 + 16 * (kp + 4 * kc)) + 144 + 16 * kc, lds_addr(&S.raw[w][48][0]));
        }
        if (b < nb - 1) roff += rstep;
    };
    // This lane's weight row 16 rq + c in one block: factors, mins of the two
    // lanes k, f16 scales of sub-blocks 2g, 2g + 1 (getScaleMinK4,
    // simd.go:1672-1677: six bits of byte 4 + j, or four bits of byte 12 + j
    // - 4 under the top two of byte 4 + j - 4) and the nibble dwords.  The
    // wave copied them itself, so they are read as soon as its own copies
    // have landed.
    struct Row {
        float d, dm, mn[2];
        h2v s, n;  // {sc_2g, sc_(2g + 1) / 16} and -1024 times them
        uint32_t nd[2], qh[2];
    };
    const uint32_t sel = g < 2 ? 4 : 12, sh0 = 16 * (g & 1), low = g < 2 ? 0x3f3fu : 0x0f0fu;
    const h2v one16 = {(_Float16)1.0f, (_Float16)0.0625f}, off16 = {(_Float16)-1024.0f, (_Float16)-64.0f};
    const h2v m1024 = {(_Float16)-1024.0f, (_Float16)-1024.0f};
    auto row_of = [&](const LnStage<Q5>& S) __attribute__((always_inline)) {
        Row r;
        const u4v h = *(const u4v*)&S.raw[w][32 + c][0];
        const uint32_t hs = *(const uint32_t*)&S.raw[w][32 + c][sel];
        r.nd[0] = *(const uint32_t*)&S.raw[w][c][4 * g];
        r.nd[1] = *(const uint32_t*)&S.raw[w][16 + c][4 * g];
        if constexpr (Q5) {
            r.qh[0] = *(const uint32_t*)&S.raw[w][48 + c][4 * kp];
            r.qh[1] = *(const uint32_t*)&S.raw[w][64 + c][4 * kp];
        }
        r.d = f16_bits_to_f32(h.x & 0xffffu);
        r.dm = factor_f16(h.x >> 16);
        r.mn[0] = (float)__builtin_amdgcn_ubfe(h.z, 8 * kp, 6);
        r.mn[1] = (float)((__builtin_amdgcn_ubfe(h.z, 8 * kp + 6, 2) << 4) | __builtin_amdgcn_ubfe(h.w, 8 * kp + 4, 4));
        const uint32_t sb = (((hs >> sh0) & low) | ((h.y >> (sh0 + 2)) & ~low)) & 0x3f3fu;
        const h2v x = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, sb, 0x04010400u));  // 1024 + sc
        r.s = __builtin_elementwise_fma(x, one16, off16);
        r.n = r.s * m1024;
        return r;
    };

    // [lane k = kp + 4 kk][token tile tt][i]
    float accF[2][4][4], accM[2][4][4];
#pragma unroll
    for (int kk = 0; kk < 2; kk++)
#pragma unroll
        for (int tt = 0; tt < 4; tt++)
#pragma unroll
            for (int i = 0; i < 4; i++) accF[kk][tt][i] = accM[kk][tt][i] = 0.0f;

    copy_raw(0, st[0]);
    copy_tokens(0, st[0]);
    copy_raw(1, st[1]);
    wait_vmem_le<kRawCopies>();
    asm volatile("" ::: "memory");
    Row row = row_of(st[0]);
    wait_lgkm0();
    lds_barrier();
    const NibMasks nm = nib_masks();
    // Block b from stage S, N the other one.  The pins and scheduling barriers
    // hold the order (the compiler would keep more operands at once than four
    // waves per SIMD have registers for).  Register 4 tt + i of an outer
    // product is token 16 tt + 4g + i.
    auto block = [&](int b, LnStage<Q5>& S, LnStage<Q5>& N) __attribute__((always_inline)) {
        copy_tokens(b + 1, N);
        copy_raw(b + 2, S);  // row b is in registers
        // LDS addresses are rebuilt from the lane each block: kept across
        // blocks they would spill
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int g = ln >> 4, c = ln & 15;
        const f16v z16 = {0.0f};
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            const f16v P = __builtin_amdgcn_mfma_f32_16x16x1f32(S.xsum[g][kp + 4 * kk][c], row.mn[kk], z16, 0, 0, 0);
#pragma unroll
            for (int tt = 0; tt < NT; tt++) {
#pragma unroll
                for (int i = 0; i < 4; i++) accM[kk][tt][i] = fmaf(row.dm, P[4 * tt + i], accM[kk][tt][i]);
                pin4(accM[kk][tt]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        const f16v dxs = __builtin_amdgcn_mfma_f32_16x16x1f32(S.xs[ln], row.d, z16, 0, 0, 0);
        // step u = (kk, tt): reads step u + 2's activations, issues its own
        // product and runs the chains of step u - 1
        const f4v z = {0.0f, 0.0f, 0.0f, 0.0f};
        auto acts = [&](int u) __attribute__((always_inline)) {
            return *(const h8v*)(S.b16 + ((u % NT * 8 + kp + 4 * (u / NT)) * 4 + g) * 256 + c * 16);
        };
        h8v bv[3], wv;
        f4v D[2];
        bv[0] = acts(0);
        bv[1] = acts(1);
#pragma unroll
        for (int u = 0; u <= 2 * NT; u++) {
            if (u < 2 * NT - 2) bv[(u + 2) % 3] = acts(u + 2);
            if (u == 0 || u == NT)
                wv = Q5 ? dequant_q5(row.nd[u / NT], row.qh[u / NT] >> (2 * g), row.s, row.n, nm)
                        : dequant_nib(row.nd[u / NT], row.s, row.n, nm);
            if (u < 2 * NT) D[u & 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bv[u % 3], wv, z, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (u > 0) {
                const int kk = (u - 1) / NT, tt = (u - 1) % NT;
#pragma unroll
                for (int i = 0; i < 4; i++)
                    accF[kk][tt][i] = fmaf(D[(u - 1) & 1][i], dxs[4 * tt + i], accF[kk][tt][i]);
                pin4(accF[kk][tt]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // block b + 1 has landed (all but the raw copy of b + 2)
        wait_vmem_le<kRawCopies>();
        asm volatile("" ::: "memory");
        row = row_of(N);
        wait_lgkm0();
        lds_barrier();
    };
#pragma unroll 1
    for (int b = 0;;) {
        block(b, st[0], st[1]);
        if (++b == nb) break;
        block(b, st[1], st[0]);
        if (++b == nb) break;
    }
    wait_vmem_le<0>();  // the last copies, never read
    lds_barrier();
    // the reference's tree: s_kp = v_kp + v_(kp + 4) here, then (s0 + s1) +
    // (s2 + s3) across the four waves of a row group, through LDS
    float* ex = (float*)dyn;  // [rq][kp][tt][i][lane]
#pragma unroll
    for (int tt = 0; tt < 4; tt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float v0 = accF[0][tt][i] - accM[0][tt][i], v1 = accF[1][tt][i] - accM[1][tt][i];
            ex[((w * 4 + tt) * 4 + i) * 64 + lane] = v0 + v1;
        }
    wait_lgkm0();
    lds_barrier();
    lanes_store(a, ex, row0, tok0, rq, kp, lane);
}

// One workgroup of 1024 threads per 64 x 64 tile.
template <size_t LDS>
static int launch_lanes(void (*kern)(PfArgs, TlMap), const PfArgs& a, hipStream_t s) {
    static_assert(LDS >= 65536 && LDS <= 160 * 1024, "the stages, and the exchange over them");
    if (!lds_opt_in((const void*)kern, LDS)) return fail(GLLM_EDEVICE, "prefill: %zu bytes of LDS were refused", LDS);
    const TlMap mp = tl_map(a.rows, a.p);
    hipLaunchKernelGGL(kern, dim3(8 * mp.tg_size * mp.rg_size), dim3(1024), LDS, s, a, mp);
    return GLLM_OK;
}

template <bool Q5>
static int launch_q4k_lanes(const PfArgs& a, hipStream_t s) {
    constexpr size_t lds = 2 * sizeof(LnStage<Q5>);
    return launch_lanes<lds>(a.p <= kHalfTok ? prefill_q4k_lanes_kernel<Q5, 2> : prefill_q4k_lanes_kernel<Q5, 4>, a, s);
}

int launch_q5k_tiled(const uint8_t* d_w, size_t rb, int rows, int blocks, const ActQ8& act, int p,
                     float* out, int out_stride, hipStream_t s) {
    if (rows <= 0 || blocks <= 0 || p <= 0) return GLLM_OK;
    if (!act.b16t || p <= kTiledMinP || (size_t)rows * rb >= ((size_t)1 << 32))
        return fail(GLLM_EINVAL, "prefill: Q5_K tiles need > %d tokens and < 4 GiB", kTiledMinP);
    GLLM_TRY(launch_q4k_lanes<true>(PfArgs{d_w, rb, rows, blocks, act, p, out, out_stride}, s));
    GLLM_HIP(hipGetLastError());
    return GLLM_OK;
}

// --- Q6_K, more than 16 activation rows: one pair of AVX2 lanes per wave ---
// q6kDotQ8KRow (kernels_amd64.s Q6KQ8QUAD, the batch-1 row kernel
// gemv_q6k_kernel) per AVX2 lane k of a 256-element block b:
//   I       = sum over the lane's 32 elements of sc(e) * code(e) * q8(e)
//             (int32; code = ql | qh << 4 in 0..63, sc the element's int8 scale)
//   o2      = fma(sc_{8+k}, 32 xs16_{8+k}, sc_k * 32 xs16_k)
//   accM[k] = fma(d_b, o2, accM[k]);  accF[k] = fma(float(I), d_b * xscale_b, accF[k])
// and tree8(accF - accM).  sc * code reaches 128 * 63, past the integers
// f16 holds exactly, so the products split at the code's two fields:
//   I = 16 * (sum sc * (code >> 4) * q8) + sum sc * (code & 15) * q8
// with |sc * (code >> 4)| <= 384 and |sc * (code & 15)| <= 1920 exact in f16
// and every partial sum of 32 products an integer below 2^24, so each of
// the two v_mfma_f32_16x16x32_f16 results is its exact integer sum and
// fma(hi, 16, lo) rounds 16 hi + lo once: float(I).
// The split of the work is prefill_q4k_lanes_kernel's: wave (rq, kp) owns 16
// rows, 64 tokens and the lanes kp and kp + 4; o2 is a product and an fma of
// outer products, two v_mfma_f32_16x16x1, and d * xscale a third.  Three VALU
// steps per product are left (fma(hi, 16, lo) and the two chains).  Weights
// need rows * rb < 4 GiB and 16-byte aligned blocks (blocks % 8 == 0).
// With the quantiser launch, 4096 x 14336 x 333 (1.5 rounds of workgroups) and
// 14336 x 4096 x 512: 473 and 490 us for 64 x 64 tiles that ran all eight
// lanes in a wave and built the A operands twice, 245 and 260 us like this.
// Bound by issue: of the SIMDs' busy cycles 64 percent VALU (190 instructions per
// wave and block, 96 of them chain steps) and 35 percent MFMA (21), a fifth of
// the latter under VALU work.
struct Q6Raw {
    uint8_t q[64][16];   // [16 part + row c]: lane kp's ql, lane kp + 4's ql, the 16 bytes with their qh
    uint8_t sc[16][16];  // [row c]
    uint32_t dw[16];     // [row c]: the dword holding d of blocks b & ~1, b | 1
};
struct Q6Stage {
    uint8_t b16[4 * 8 * 4 * 256];  // [token tile][lane k][group g][token c][8 halves]
    float x16[4][kTlTok][4];       // [16-group / 4][token][16-group % 4] xs16
    float xs[kTlTok];
    Q6Raw raw[16];                 // [wave]
};

// A code field of two bytes (0 and 2, or 1 and 3) at bits 4 .. under f16
// exponent bits of 64 reads 64 + field.
struct Q6Masks {  // held in registers, as NibMasks
    uint32_t nib, lo2, hi2, exp;
};

// f16 operands of a lane (g, c)'s 8 codes of one AVX2 lane: quads 2g (scale
// S[0]) and 2g + 1 (S[1]) from ql dwords 2 (g / 2), 2 (g / 2) + 1 and qh dword
// g / 2, the nibble (bit pairs) 4 (g % 2) up.
__device__ __forceinline__ h8v q6_lows(uint2 ql, h2v S, int g, const Q6Masks& m) {
    const uint32_t s0 = 4 - 4 * (g & 1), s1 = 4 + 4 * (g & 1);  // the nibble to bits 4-7
    const h2v m64 = {(_Float16)-64.0f, (_Float16)-64.0f};
    const h2v N = S * m64;  // (64 + q) S + N is exact
    const h2v sl = {S[0], S[0]}, nl = {N[0], N[0]}, sh = {S[1], S[1]}, nh = {N[1], N[1]};
    const h2v p0 = __builtin_bit_cast(h2v, ((ql.x << s0) & m.nib) | m.exp), p1 = __builtin_bit_cast(h2v, ((ql.x >> s1) & m.nib) | m.exp);
    const h2v p2 = __builtin_bit_cast(h2v, ((ql.y << s0) & m.nib) | m.exp), p3 = __builtin_bit_cast(h2v, ((ql.y >> s1) & m.nib) | m.exp);
    const h2v a0 = __builtin_elementwise_fma(p0, sl, nl), a1 = __builtin_elementwise_fma(p1, sl, nl);
    const h2v a2 = __builtin_elementwise_fma(p2, sh, nh), a3 = __builtin_elementwise_fma(p3, sh, nh);
    return h8v{a0[0], a0[1], a1[0], a1[1], a2[0], a2[1], a3[0], a3[1]};
}
__device__ __forceinline__ h8v q6_highs(uint32_t qh, h2v S, int g, const Q6Masks& m) {
    const uint32_t s0 = 4 - 4 * (g & 1), s1 = 4 + 4 * (g & 1);
    const h2v quarter = {(_Float16)1.0f, (_Float16)0.25f}, m64 = {(_Float16)-64.0f, (_Float16)-64.0f};
    const h2v T = S * quarter, N = T * m64;  // quad 2g + 1's field sits two bits higher: 64 + 4 q
    const h2v sl = {T[0], T[0]}, nl = {N[0], N[0]}, sh = {T[1], T[1]}, nh = {N[1], N[1]};
    const uint32_t y0 = qh << s0, y1 = qh >> s1;
    const h2v p0 = __builtin_bit_cast(h2v, (y0 & m.lo2) | m.exp), p1 = __builtin_bit_cast(h2v, (y1 & m.lo2) | m.exp);
    const h2v p2 = __builtin_bit_cast(h2v, (y0 & m.hi2) | m.exp), p3 = __builtin_bit_cast(h2v, (y1 & m.hi2) | m.exp);
    const h2v a0 = __builtin_elementwise_fma(p0, sl, nl), a1 = __builtin_elementwise_fma(p1, sl, nl);
    const h2v a2 = __builtin_elementwise_fma(p2, sh, nh), a3 = __builtin_elementwise_fma(p3, sh, nh);
    return h8v{a0[0], a0[1], a1[0], a1[1], a2[0], a2[1], a3[0], a3[1]};
}

template <int NT>
__global__ __launch_bounds__(1024) void prefill_q6k_lanes_kernel(PfArgs a, TlMap mp) {
    extern __shared__ __attribute__((aligned(16))) uint8_t dyn[];
    Q6Stage* const st = (Q6Stage*)dyn;
    const int id = blockIdx.x, xcd = id & 7, local = id >> 3;
    const int lt = local % mp.tg_size, lrow = local / mp.tg_size;
    const int ttile = (xcd % mp.h) * mp.tg_size + lt, rtile = (xcd / mp.h) * mp.rg_size + lrow;
    if (lrow >= mp.rg_size || ttile >= mp.tok_tiles || rtile >= mp.row_tiles) return;  // whole workgroup
    const int row0 = rtile * kTlRows, tok0 = ttile * kTlTok, tile0 = tok0 / 16;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, c = lane & 15;
    const int kp = w & 3, rq = w >> 2;
    const int nb = a.blocks;

    // Copies of one block's tokens: two 1 KB pieces of B16 (as in the Q4_K
    // kernel), the tokens' xs16 (waves 0-3, four 16-groups each) and xscales
    // (wave 4)
    const int last = a.act.tiles - 1, tok = min(tok0 + lane, a.p - 1);
    const size_t bstep = (size_t)a.act.tiles * 8192;
    const uint8_t* bsrc = (const uint8_t*)a.act.b16t + (size_t)min(tile0 + rq, last) * 8192 + 2048 * kp;
    const uint32_t xoff = w < 4 ? (uint32_t)tok * nb * 64 + 16 * w : (uint32_t)tok * nb * 4;
    auto copy_tokens = [&](int b, Q6Stage& S) __attribute__((always_inline)) {
        b = min(b, nb - 1);
        const uint8_t* src = bsrc + b * bstep;
        const uint32_t dst = lds_addr(S.b16 + rq * 8192 + 2048 * kp);
        lds_copy16_s(src, 16 * lane, dst);
        lds_copy16_s(src + 1024, 16 * lane, dst + 1024);
        if (w < 4) lds_copy16_s(a.act.xs16 + (size_t)b * 16, xoff, lds_addr(&S.x16[w][0][0]));
        else if (w == 4) lds_copy4_s(a.act.xscale + b, xoff, lds_addr(&S.xs[0]));
    };
    // The wave's rows: three copies
    const uint32_t rbase = (uint32_t)min(row0 + 16 * rq + c, a.rows - 1) * (uint32_t)a.rb;
    const uint32_t qoff = rbase + (g < 2 ? 16 * (kp + 4 * g) : 128 + 16 * ((kp >> 1) + 2 * (g - 2)));
    auto copy_raw = [&](int b, Q6Stage& S) __attribute__((always_inline)) {
        b = min(b, nb - 1);
        const uint8_t* src = a.w + (size_t)b * 208;
        lds_copy16_s(src, qoff, lds_addr(&S.raw[w].q[0][0]));
        if (lane < 16) {
            lds_copy16_s(src + 192, rbase, lds_addr(&S.raw[w].sc[0][0]));
            lds_copy4_s(a.w, rbase + (uint32_t)(nb * 208 + (b & ~1) * 2), lds_addr(&S.raw[w].dw[0]));
        }
    };

    // [lane k = kp + 4 kk][token tile tt][i]
    float accF[2][4][4], accM[2][4][4];
#pragma unroll
    for (int kk = 0; kk < 2; kk++)
#pragma unroll
        for (int tt = 0; tt < 4; tt++)
#pragma unroll
            for (int i = 0; i < 4; i++) accF[kk][tt][i] = accM[kk][tt][i] = 0.0f;

    Q6Masks m{0x00f000f0u, 0x00300030u, 0x00c000c0u, 0x54005400u};
    asm("" : "+s"(m.nib), "+s"(m.lo2), "+s"(m.hi2), "+v"(m.exp));
    const h2v m1152 = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    copy_raw(0, st[0]);
    copy_tokens(0, st[0]);
    copy_raw(1, st[1]);
    wait_vmem_le<3>();
    lds_barrier();
    // Block b from stage S, N the other one; register 4 tt + i of an outer
    // product is token 16 tt + 4g + i
    auto block = [&](int b, Q6Stage& S, Q6Stage& N) __attribute__((always_inline)) {
        copy_tokens(b + 1, N);
        const Q6Raw& R = S.raw[w];
        // LDS addresses are rebuilt from the lane each block: kept across
        // blocks they would spill
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int g = ln >> 4, c = ln & 15, lane = ln;
        const int8_t* rsc = (const int8_t*)R.sc[c];
        const uint32_t sv = *(const uint32_t*)&R.sc[c][4 * g] ^ 0x80808080u;  // s + 128
        const float d = factor_f16(R.dw[c] >> (16 * (b & 1)));
        const f16v z16 = {0.0f};
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            const float x0 = S.x16[kk][lane][kp] * 32.0f;      // ScaleF32(xs, 32)
            const float x8 = S.x16[2 + kk][lane][kp] * 32.0f;
            const float sk = (float)rsc[kp + 4 * kk], sk8 = (float)rsc[8 + kp + 4 * kk];
            f16v P = __builtin_amdgcn_mfma_f32_16x16x1f32(x0, sk, z16, 0, 0, 0);  // VMULPS
            P = __builtin_amdgcn_mfma_f32_16x16x1f32(x8, sk8, P, 0, 0, 0);        // VFMADD231PS
#pragma unroll
            for (int tt = 0; tt < NT; tt++) {
#pragma unroll
                for (int i = 0; i < 4; i++) accM[kk][tt][i] = fmaf(d, P[4 * tt + i], accM[kk][tt][i]);
                pin4(accM[kk][tt]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        const f16v dxs = __builtin_amdgcn_mfma_f32_16x16x1f32(S.xs[lane], d, z16, 0, 0, 0);
        // step u = (kk, tt); the next step's activations are read ahead
        const f4v z = {0.0f, 0.0f, 0.0f, 0.0f};
        auto acts = [&](int u) __attribute__((always_inline)) {
            return *(const h8v*)(S.b16 + ((u % NT * 8 + kp + 4 * (u / NT)) * 4 + g) * 256 + c * 16);
        };
        h8v bv[2], wl, wh;
        bv[0] = acts(0);
#pragma unroll
        for (int u = 0; u < 2 * NT; u++) {
            const int kk = u / NT, tt = u % NT;
            if (u < 2 * NT - 1) bv[(u + 1) & 1] = acts(u + 1);
            if (tt == 0) {
                const uint2 ql = *(const uint2*)&R.q[16 * kk + c][8 * (g >> 1)];
                const uint32_t qh = *(const uint32_t*)&R.q[32 + 16 * kk + c][8 * (kp & 1) + 4 * (g >> 1)];
                const h2v sc = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, sv, kk ? 0x04030401u : 0x04020400u)) + m1152;
                wl = q6_lows(ql, sc, g, m);
                wh = q6_highs(qh, sc, g, m);
            }
            const f4v lo = __builtin_amdgcn_mfma_f32_16x16x32_f16(bv[u & 1], wl, z, 0, 0, 0);
            const f4v hi = __builtin_amdgcn_mfma_f32_16x16x32_f16(bv[u & 1], wh, z, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float iv = fmaf(hi[i], 16.0f, lo[i]);  // float(I)
                accF[kk][tt][i] = fmaf(iv, dxs[4 * tt + i], accF[kk][tt][i]);
            }
            pin4(accF[kk][tt]);
            __builtin_amdgcn_sched_barrier(0);
            // the wave's last read of its raw rows has returned: refill their
            // slot two blocks ahead
            if (u == NT) copy_raw(b + 2, S);
        }
        wait_vmem_le<3>();  // block b + 1 has landed (all but the raw copies of b + 2)
        wait_lgkm0();
        lds_barrier();
    };
#pragma unroll 1
    for (int b = 0;;) {
        block(b, st[0], st[1]);
        if (++b == nb) break;
        block(b, st[1], st[0]);
        if (++b == nb) break;
    }
    wait_vmem_le<0>();  // the last copies, never read
    lds_barrier();
    // the tree, as in the Q4_K kernel
    float* ex = (float*)dyn;  // [rq][kp][tt][i][lane]
#pragma unroll
    for (int tt = 0; tt < 4; tt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float v0 = accF[0][tt][i] - accM[0][tt][i], v1 = accF[1][tt][i] - accM[1][tt][i];
            ex[((w * 4 + tt) * 4 + i) * 64 + lane] = v0 + v1;
        }
    wait_lgkm0();
    lds_barrier();
    lanes_store(a, ex, row0, tok0, rq, kp, lane);
}

int launch_q6k_tiled(const uint8_t* d_w, size_t rb, int rows, int blocks, const ActQ8& act, int p,
                     float* out, int out_stride, hipStream_t s) {
    if (rows <= 0 || blocks <= 0 || p <= 0) return GLLM_OK;
    if (!act.b16t || p <= kTiledMinP || blocks % 8 || (size_t)rows * rb >= ((size_t)1 << 32) ||
        (size_t)p * blocks * 64 >= ((size_t)1 << 32))
        return fail(GLLM_EINVAL, "prefill: Q6_K tiles need > %d tokens, blocks %% 8 == 0, < 4 GiB of weight and of sums",
                    kTiledMinP);
    PfArgs a{d_w, rb, rows, blocks, act, p, out, out_stride};
    constexpr size_t lds = 2 * sizeof(Q6Stage);
    GLLM_TRY((launch_lanes<lds>(p <= kHalfTok ? prefill_q6k_lanes_kernel<2> : prefill_q6k_lanes_kernel<4>, a, s)));
    GLLM_HIP(hipGetLastError());
    return GLLM_OK;
}

// --- Q8_0, more than 16 activation rows: one pair of AVX2 lanes per wave ----
// q8_0DotQ8KRow (kernels_amd64.s Q80CHUNK) per AVX2 lane k of a 256-element
// group: for its eight 32-value blocks q in order
//   acc12 = fma(d_q, float(I_qk), acc12)   I_qk: the exact dot of the lane's
//                                           4 weight and 4 activation bytes
// then acc11[k] = fma(xscale, acc12, acc11[k]) and tree8(acc11).  The
// float chain over q is nine VALU steps per product and lane; the dots in
// front of it are matrix products with K = 4, so v_mfma_f32_16x16x4 (f16,
// four blocks) delivers float(I) for four q of a 16 x 16 tile at once, exact
// (integers below 2^17) where the VALU takes a v_dot4_i32_i8 and a
// conversion each.
// The split of the work is prefill_q4k_lanes_kernel's: wave (rq, kp) owns 16
// rows, 64 tokens and the lanes kp and kp + 4.  A lane's 16 bytes of B16 hold
// blocks 2g (first four halves) and 2g + 1, so the even and the odd q are one
// instruction each.
// With the quantiser launch, 14336 x 4096 x 512: 718 us for 64 x 64 tiles on
// the vector units (25 VALU operations per lane product), 305 us like this.
// Bound by the VALU, 93 percent of the SIMDs' busy cycles; two thirds of the
// matrix instructions' cycles run under it.
struct Q80Raw {
    uint8_t q[64][16];  // [32 (k / 4) + 16 half + row c]
    uint8_t d[16][16];  // [row c]: eight f16 scales
};
struct Q80Stage {
    uint8_t b16[4 * 8 * 4 * 256];  // [token tile][lane k][group g][token c][8 halves]
    float xs[kTlTok];
    Q80Raw raw[16];                // [wave]
};
typedef _Float16 h4v __attribute__((ext_vector_type(4)));

template <int NT>
__global__ __launch_bounds__(1024) void prefill_q8_0_lanes_kernel(PfArgs a, TlMap mp) {
    extern __shared__ __attribute__((aligned(16))) uint8_t dyn[];
    Q80Stage* const st = (Q80Stage*)dyn;
    const int id = blockIdx.x, xcd = id & 7, local = id >> 3;
    const int lt = local % mp.tg_size, lrow = local / mp.tg_size;
    const int ttile = (xcd % mp.h) * mp.tg_size + lt, rtile = (xcd / mp.h) * mp.rg_size + lrow;
    if (lrow >= mp.rg_size || ttile >= mp.tok_tiles || rtile >= mp.row_tiles) return;  // whole workgroup
    const int row0 = rtile * kTlRows, tok0 = ttile * kTlTok, tile0 = tok0 / 16;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kp = w & 3, rq = w >> 2;
    const int nb = a.blocks;

    // Copies of one group's tokens: two 1 KB pieces of B16 (as in the Q4_K
    // kernel) and the xscales (wave 0)
    const int last = a.act.tiles - 1;
    const size_t bstep = (size_t)a.act.tiles * 8192;
    const uint8_t* bsrc = (const uint8_t*)a.act.b16t + (size_t)min(tile0 + rq, last) * 8192 + 2048 * kp;
    const uint32_t xoff = (uint32_t)min(tok0 + lane, a.p - 1) * nb * 4;
    auto copy_tokens = [&](int b, Q80Stage& S) __attribute__((always_inline)) {
        b = min(b, nb - 1);
        const uint8_t* src = bsrc + b * bstep;
        const uint32_t dst = lds_addr(S.b16 + rq * 8192 + 2048 * kp);
        lds_copy16_s(src, 16 * lane, dst);
        lds_copy16_s(src + 1024, 16 * lane, dst + 1024);
        if (w == 0) lds_copy4_s(a.act.xscale + b, xoff, lds_addr(&S.xs[0]));
    };
    // The wave's rows: two copies
    const uint32_t rbase = (uint32_t)min(row0 + 16 * rq + (lane & 15), a.rows - 1) * (uint32_t)a.rb;
    const uint32_t qoff = rbase + 16 + 32 * (kp + 4 * (lane >> 5)) + 16 * ((lane >> 4) & 1);
    auto copy_raw = [&](int b, Q80Stage& S) __attribute__((always_inline)) {
        const uint8_t* src = a.w + (size_t)min(b, nb - 1) * 272;
        lds_copy16_s(src, qoff, lds_addr(&S.raw[w].q[0][0]));
        if (lane < 16) lds_copy16_s(src, rbase, lds_addr(&S.raw[w].d[0][0]));
    };

    float acc[2][4][4];  // acc11 of [lane k = kp + 4 kk][token tile tt][i]
#pragma unroll
    for (int kk = 0; kk < 2; kk++)
#pragma unroll
        for (int tt = 0; tt < 4; tt++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[kk][tt][i] = 0.0f;

    uint32_t bytes = 0x00ff00ffu, exp = 0x64006400u;
    asm("" : "+s"(bytes), "+v"(exp));
    const h2v m1152 = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    // a dword of int8 as f16, bytes 0, 2, 1, 3: 1024 + (v + 128) - 1152
    auto halves = [&](uint32_t v) __attribute__((always_inline)) {
        v ^= 0x80808080u;
        const h2v p0 = __builtin_bit_cast(h2v, (v & bytes) | exp) + m1152;
        const h2v p1 = __builtin_bit_cast(h2v, ((v >> 8) & bytes) | exp) + m1152;
        return h4v{p0[0], p0[1], p1[0], p1[1]};
    };

    copy_raw(0, st[0]);
    copy_tokens(0, st[0]);
    copy_raw(1, st[1]);
    wait_vmem_le<2>();
    lds_barrier();
    auto block = [&](int b, Q80Stage& S, Q80Stage& N) __attribute__((always_inline)) {
        copy_tokens(b + 1, N);
        int ln = lane;  // LDS addresses are rebuilt each block: kept across blocks they would spill
        asm volatile("" : "+v"(ln));
        const int g = ln >> 4, c = ln & 15;
        const Q80Raw& R = S.raw[w];
        const u4v dh = *(const u4v*)&R.d[c][0];
        float d[8];
#pragma unroll
        for (int q = 0; q < 8; q++) d[q] = factor_f16(dh[q >> 1] >> (16 * (q & 1)));
        // step u = (kk, tt): token 16 tt + 4g + i, weight row 16 rq + c
        auto acts = [&](int u) __attribute__((always_inline)) {
            return *(const h8v*)(S.b16 + ((u % NT * 8 + kp + 4 * (u / NT)) * 4 + g) * 256 + c * 16);
        };
        h8v bv[2];
        h4v we, wo;
        bv[0] = acts(0);
#pragma unroll
        for (int u = 0; u < 2 * NT; u++) {
            const int kk = u / NT, tt = u % NT;
            if (u < 2 * NT - 1) bv[(u + 1) & 1] = acts(u + 1);
            if (tt == 0) {
                const uint2 v = *(const uint2*)&R.q[32 * kk + 16 * (g >> 1) + c][8 * (g & 1)];
                we = halves(v.x);
                wo = halves(v.y);
            }
            const f4v xs = *(const f4v*)&S.xs[16 * tt + 4 * g];
            const h8v x = bv[u & 1];
            const f16v z16 = {0.0f};
            const f16v E = __builtin_amdgcn_mfma_f32_16x16x4f16(h4v{x[0], x[1], x[2], x[3]}, we, z16, 0, 0, 0);
            const f16v O = __builtin_amdgcn_mfma_f32_16x16x4f16(h4v{x[4], x[5], x[6], x[7]}, wo, z16, 0, 0, 0);
            float y[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int q = 0; q < 4; q++) {
#pragma unroll
                for (int i = 0; i < 4; i++) y[i] = fmaf(E[4 * q + i], d[2 * q], y[i]);  // VFMADD231PS
#pragma unroll
                for (int i = 0; i < 4; i++) y[i] = fmaf(O[4 * q + i], d[2 * q + 1], y[i]);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) acc[kk][tt][i] = fmaf(y[i], xs[i], acc[kk][tt][i]);
            pin4(acc[kk][tt]);
            __builtin_amdgcn_sched_barrier(0);
            // the wave's last read of its raw rows has returned: refill their
            // slot two groups ahead
            if (u == NT) copy_raw(b + 2, S);
        }
        wait_vmem_le<2>();  // group b + 1 has landed (all but the raw copies of b + 2)
        wait_lgkm0();
        lds_barrier();
    };
#pragma unroll 1
    for (int b = 0;;) {
        block(b, st[0], st[1]);
        if (++b == nb) break;
        block(b, st[1], st[0]);
        if (++b == nb) break;
    }
    wait_vmem_le<0>();  // the last copies, never read
    lds_barrier();
    float* ex = (float*)dyn;  // [rq][kp][tt][i][lane]
#pragma unroll
    for (int tt = 0; tt < 4; tt++)
#pragma unroll
        for (int i = 0; i < 4; i++) ex[((w * 4 + tt) * 4 + i) * 64 + lane] = acc[0][tt][i] + acc[1][tt][i];
    wait_lgkm0();
    lds_barrier();
    lanes_store(a, ex, row0, tok0, rq, kp, lane);
}

int launch_q8_0_tiled(const uint8_t* d_w, size_t rb, int rows, int blocks, const ActQ8& act, int p,
                      float* out, int out_stride, hipStream_t s) {
    if (rows <= 0 || blocks <= 0 || p <= 0) return GLLM_OK;
    if (!act.b16t || p <= kTiledMinP || (size_t)rows * rb >= ((size_t)1 << 32))
        return fail(GLLM_EINVAL, "prefill: Q8_0 tiles need > %d tokens and < 4 GiB", kTiledMinP);
    PfArgs a{d_w, rb, rows, blocks, act, p, out, out_stride};
    constexpr size_t lds = 2 * sizeof(Q80Stage);
    GLLM_TRY((launch_lanes<lds>(p <= kHalfTok ? prefill_q8_0_lanes_kernel<2> : prefill_q8_0_lanes_kernel<4>, a, s)));
    GLLM_HIP(hipGetLastError());
    return GLLM_OK;
}

// --- Q4_0, more than 16 activation rows: one pair of AVX2 lanes per wave ----
// q4_0DotQ8KRow (kernels_amd64.s:679-732) per 32-value block q:
//   accF[k] = fma(d_q * xscale, float(I_qk), accF[k])   I_qk: the exact dot of the lane's
//                                                       4 codes and 4 activation bytes
//   accS    = fma(-8, d_q * xsum_q, accS)               one chain per row
// and tree8(accF) + accS.  The split of the work and the dots are
// prefill_q8_0_lanes_kernel's; a wave's lanes kp and kp + 4 are the low and
// the high nibbles of the same 32 bytes.  d_q * xscale of four q is one
// v_mfma_f32_16x16x1 (block j of the four: q = 2j, or 2j + 1) per token tile,
// for both lanes, and the offset chains of token tile kp go with wave
// (rq, kp), which stores that tile.
// With the quantiser launch, the row kernels eight tokens at a time / this:
// 14336 x 4096 x 512 3304 / 441 us, 4096 x 14336 x 333 3914 / 388, 4096 x 4096
// x 64 243 / 56, 14336 x 4096 x 24 154 / 41; where 16 workgroups are all there
// is, 1000 x 14336 x 17 133 / 115 and 1000 x 4096 x 17 49 / 38 us (179 and 56
// with the token tiles past p computed too).  Bound by issue: per wave and
// block 288 chain steps and 26 matrix instructions.
struct Q40Stage {
    uint8_t b16[4 * 8 * 4 * 256];  // [token tile][lane k][group g][token c][8 halves]
    float xsum[4][8][16];          // [token tile][32-block q][token c]
    float xs[kTlTok];
    uint8_t raw[16][48][16];       // [wave]: nibbles [16 half + row c], eight f16 scales [32 + row c]
};

__global__ __launch_bounds__(1024) void prefill_q4_0_lanes_kernel(PfArgs a, TlMap mp) {
    extern __shared__ __attribute__((aligned(16))) uint8_t dyn[];
    Q40Stage* const st = (Q40Stage*)dyn;
    const int id = blockIdx.x, xcd = id & 7, local = id >> 3;
    const int lt = local % mp.tg_size, lrow = local / mp.tg_size;
    const int ttile = (xcd % mp.h) * mp.tg_size + lt, rtile = (xcd / mp.h) * mp.rg_size + lrow;
    if (lrow >= mp.rg_size || ttile >= mp.tok_tiles || rtile >= mp.row_tiles) return;  // whole workgroup
    const int row0 = rtile * kTlRows, tok0 = ttile * kTlTok, tile0 = tok0 / 16;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kp = w & 3, rq = w >> 2;
    const int nb = a.blocks, left = a.p - tok0;  // token tiles past p are left out

    // Copies of one block's tokens, as in the Q4_K kernel
    const int last = a.act.tiles - 1;
    const size_t bstep = (size_t)a.act.tiles * 8192;
    const uint8_t* bsrc = (const uint8_t*)a.act.b16t + (size_t)min(tile0 + rq, last) * 8192 + 2048 * kp;
    const uint32_t xoff = w < 2 ? (uint32_t)(min(tile0 + 2 * w + (lane >> 5), last) * 512 + 16 * (lane & 31))
                                : (uint32_t)min(tok0 + lane, a.p - 1) * nb * 4;
    auto copy_tokens = [&](int b, Q40Stage& S) __attribute__((always_inline)) {
        b = min(b, nb - 1);
        const uint8_t* src = bsrc + b * bstep;
        const uint32_t dst = lds_addr(S.b16 + rq * 8192 + 2048 * kp);
        lds_copy16_s(src, 16 * lane, dst);
        lds_copy16_s(src + 1024, 16 * lane, dst + 1024);
        if (w < 2) lds_copy16_s(a.act.xs32t + (size_t)b * a.act.tiles * 128, xoff, lds_addr(&S.xsum[2 * w][0][0]));
        else if (w == 2) lds_copy4_s(a.act.xscale + b, xoff, lds_addr(&S.xs[0]));
    };
    // The wave's rows: one copy
    const uint32_t roff = (uint32_t)min(row0 + 16 * rq + (lane & 15), a.rows - 1) * (uint32_t)a.rb +
                          (lane < 32 ? 16 + 32 * kp + 16 * (lane >> 4) : 0);
    auto copy_raw = [&](int b, Q40Stage& S) __attribute__((always_inline)) {
        if (lane < 48) lds_copy16_s(a.w + (size_t)min(b, nb - 1) * 144, roff, lds_addr(&S.raw[w][0][0]));
    };

    float acc[2][4][4];  // accF of [lane k = kp + 4 kk][token tile tt][i]
    f4v off = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kk = 0; kk < 2; kk++)
#pragma unroll
        for (int tt = 0; tt < 4; tt++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[kk][tt][i] = 0.0f;

    uint32_t nib = 0x000f000fu, exp = 0x64006400u;
    asm("" : "+s"(nib), "+v"(exp));
    const h2v m1024 = {(_Float16)-1024.0f, (_Float16)-1024.0f};
    // the low nibbles of a dword as f16, bytes 0, 2, 1, 3: 1024 + code - 1024
    auto halves = [&](uint32_t v) __attribute__((always_inline)) {
        const h2v p0 = __builtin_bit_cast(h2v, (v & nib) | exp) + m1024;
        const h2v p1 = __builtin_bit_cast(h2v, ((v >> 8) & nib) | exp) + m1024;
        return h4v{p0[0], p0[1], p1[0], p1[1]};
    };

    copy_raw(0, st[0]);
    copy_tokens(0, st[0]);
    copy_raw(1, st[1]);
    wait_vmem_le<1>();
    lds_barrier();
    auto block = [&](int b, Q40Stage& S, Q40Stage& N) __attribute__((always_inline)) {
        copy_tokens(b + 1, N);
        int ln = lane;  // LDS addresses are rebuilt each block: kept across blocks they would spill
        asm volatile("" : "+v"(ln));
        const int g = ln >> 4, c = ln & 15;
        // this lane's codes and scales: 32-blocks 2g, 2g + 1 of row c
        const uint2 v = *(const uint2*)&S.raw[w][16 * (g >> 1) + c][8 * (g & 1)];
        const uint32_t dd = *(const uint32_t*)&S.raw[w][32 + c][4 * g];
        wait_lgkm0();
        copy_raw(b + 2, S);  // the wave's rows are in registers
        const float de = f16_bits_to_f32(dd & 0xffffu), dn = f16_bits_to_f32(dd >> 16);
        const f16v z16 = {0.0f};
        {
            const f16v E = __builtin_amdgcn_mfma_f32_16x16x1f32(S.xsum[kp][2 * g][c], de, z16, 0, 0, 0);
            const f16v O = __builtin_amdgcn_mfma_f32_16x16x1f32(S.xsum[kp][2 * g + 1][c], dn, z16, 0, 0, 0);
#pragma unroll
            for (int q = 0; q < 4; q++) {
#pragma unroll
                for (int i = 0; i < 4; i++) off[i] = fmaf(-8.0f, E[4 * q + i], off[i]);  // VFMADD231SS
#pragma unroll
                for (int i = 0; i < 4; i++) off[i] = fmaf(-8.0f, O[4 * q + i], off[i]);
            }
            asm volatile("" : "+v"(off));
        }
        __builtin_amdgcn_sched_barrier(0);
        // token 16 tt + 4g + i, weight row 16 rq + c
#pragma unroll
        for (int tt = 0; tt < 4; tt++) {
            if (16 * tt >= left) break;
            const float xs = S.xs[16 * tt + c];
            const f16v dE = __builtin_amdgcn_mfma_f32_16x16x1f32(xs, de, z16, 0, 0, 0);  // VMULSS
            const f16v dO = __builtin_amdgcn_mfma_f32_16x16x1f32(xs, dn, z16, 0, 0, 0);
#pragma unroll
            for (int kk = 0; kk < 2; kk++) {
                const h8v x = *(const h8v*)(S.b16 + ((tt * 8 + kp + 4 * kk) * 4 + g) * 256 + c * 16);
                const f16v E = __builtin_amdgcn_mfma_f32_16x16x4f16(h4v{x[0], x[1], x[2], x[3]}, halves(v.x >> (4 * kk)), z16, 0, 0, 0);
                const f16v O = __builtin_amdgcn_mfma_f32_16x16x4f16(h4v{x[4], x[5], x[6], x[7]}, halves(v.y >> (4 * kk)), z16, 0, 0, 0);
#pragma unroll
                for (int q = 0; q < 4; q++) {
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[kk][tt][i] = fmaf(E[4 * q + i], dE[4 * q + i], acc[kk][tt][i]);  // VFMADD231PS
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[kk][tt][i] = fmaf(O[4 * q + i], dO[4 * q + i], acc[kk][tt][i]);
                }
                pin4(acc[kk][tt]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        wait_vmem_le<1>();  // block b + 1 has landed (all but the raw copy of b + 2)
        wait_lgkm0();
        lds_barrier();
    };
#pragma unroll 1
    for (int b = 0;;) {
        block(b, st[0], st[1]);
        if (++b == nb) break;
        block(b, st[1], st[0]);
        if (++b == nb) break;
    }
    wait_vmem_le<0>();  // the last copies, never read
    lds_barrier();
    float* ex = (float*)dyn;  // [rq][kp][tt][i][lane]
#pragma unroll
    for (int tt = 0; tt < 4; tt++)
#pragma unroll
        for (int i = 0; i < 4; i++) ex[((w * 4 + tt) * 4 + i) * 64 + lane] = acc[0][tt][i] + acc[1][tt][i];
    wait_lgkm0();
    lds_barrier();
    lanes_store<true>(a, ex, row0, tok0, rq, kp, lane, off);
}

int launch_q4_0_tiled(const uint8_t* d_w, size_t rb, int rows, int blocks, const ActQ8& act, int p,
                      float* out, int out_stride, hipStream_t s) {
    if (rows <= 0 || blocks <= 0 || p <= 0) return GLLM_OK;
    if (!act.b16t || p <= kTiledMinP || (size_t)rows * rb >= ((size_t)1 << 32))
        return fail(GLLM_EINVAL, "prefill: Q4_0 tiles need > %d tokens and < 4 GiB", kTiledMinP);
    PfArgs a{d_w, rb, rows, blocks, act, p, out, out_stride};
    constexpr size_t lds = 2 * sizeof(Q40Stage);
    GLLM_TRY((launch_lanes<lds>(prefill_q4_0_lanes_kernel, a, s)));
    GLLM_HIP(hipGetLastError());
    return GLLM_OK;
}

// --- 2 to 16 activation rows: one pair of AVX2 lanes per wave ---------------
// A decode batch reads the weights once for few tokens, so a workgroup is 16
// rows, split over 4 / KP waves of KP lane pairs (kp, kp + 4), and every wave
// streams what it needs of a block by itself, kSmRing blocks ahead in LDS: 16
// rows' nibbles of its lanes, their headers, and its records of the
// activations (small_rec: f16 operands and sums).  No wave waits for another
// before the final tree, so there is no barrier in the loop.
// KP: four waves take 16-byte pieces of each 128-byte weight line at
// different times, two waves of two pairs each fetch it less often: at 14336 x
// 4096 and 8 tokens a launch makes 745 thousand L2 reads in 14.4 us, with one pair
// per wave 857 thousand in 16.0 us.  Where rows are few and waves scarce one
// pair per wave is faster.
// Up to 8 tokens (PT = 8) both lanes share one MFMA tile: D rows 0-7 hold lane
// kp's eight tokens and rows 8-15 lane kp + 4's, two MFMAs accumulating into
// it with the other lane's A rows zero (read from a zeroed LDS row; every sum
// is an exact integer below 2^24), so the chains run on full registers.
// Q6_K has the code's two fields and xs16, as in prefill_q6k_lanes_kernel.
// With the quantiser launch (3-4 us of it): Q4_K 14336 x 4096 at 8 tokens 21.0
// us for 64-row tiles staged per block, 16.5 like this; 4096 x 14336 at 3 / 8 /
// 16 tokens 31.8 / 23.4 / 37.8 -> 17.5 / 18.0 / 21.2 us; Q6_K 4096 x 14336 at 5
// / 16 tokens 40.4 / 107 -> 26.3 / 30.9 us for the row kernels.
constexpr int kSmRing = 4;

template <int PT, bool Q6, int KP>
struct SmSlot {
    // Q6Raw, or nibbles [32 j + 16 (k / 4) + row c of pair j] and headers [row c]
    static constexpr int kRaw = Q6 ? 64 * 16 + 16 * 16 + 16 * 4 : (32 * KP + 16) * 16;
    uint8_t raw[kRaw];
    uint8_t rec[KP][PT * 128 + PT * 28];
};
template <int PT, bool Q6, int KP>
struct SmLds {
    SmSlot<PT, Q6, KP> ring[4 / KP][kSmRing];  // [wave]
    uint8_t zero[16];
    float ex[4][64][4];
};

// Weights of one type and width, their row tiles end to end in one grid: Q/K/V
// of 4096 + 1024 + 1024 rows x 4096 at 5 tokens take 10.5 us with the quantiser,
// 21.8 with a launch each and 14.6 on the row kernels' one launch.
template <int PT, bool Q6, int KP>
__global__ __launch_bounds__(256 / KP) void small_lanes_kernel(SmallJob job) {
    static_assert(KP == 1 || !Q6, "two pairs per wave: Q4_K");
    int wi = 0;
    while (wi + 1 < job.n && (int)blockIdx.x >= job.wg_begin[wi + 1]) wi++;
    const uint8_t* const W = job.w[wi];
    const int rows = job.rows[wi], nb = job.blocks;
    constexpr int KK = PT == 8 ? 1 : 2;  // MFMA tiles of a pair: both lanes in one, or one each
    __shared__ __attribute__((aligned(16))) SmLds<PT, Q6, KP> L;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kp = KP * wave;  // the wave's first pair
    const int g = lane >> 4, c = lane & 15;
    const int row0 = ((int)blockIdx.x - job.wg_begin[wi]) * 16;
    if (threadIdx.x < 4) ((uint32_t*)L.zero)[threadIdx.x] = 0;
    const uint32_t rbase = (uint32_t)min(row0 + c, rows - 1) * (uint32_t)job.rb;
    uint32_t roff;  // the lane's source in the first raw copy
    if constexpr (Q6) roff = rbase + (g < 2 ? 16 * (kp + 4 * g) : 128 + 16 * ((kp >> 1) + 2 * (g - 2)));
    else if constexpr (KP == 1) roff = rbase + (g < 2 ? 16 * nb + 16 * (kp + 4 * g) : 0);
    else roff = rbase + 16 * nb + 16 * (kp + (g >> 1) + 4 * (g & 1));
    constexpr int REC = PT * 128 + PT * 28, RECS = KP * REC;
    constexpr int kCopies = (Q6 ? 3 : KP) + RECS / 1024 + 1;  // per block
    const uint8_t* rec = job.rec + (size_t)kp * REC;
    auto copy = [&](int b, SmSlot<PT, Q6, KP>& S) __attribute__((always_inline)) {
        b = min(b, nb - 1);
        const uint32_t raw = lds_addr(S.raw), dst = lds_addr(S.rec[0]);
        if constexpr (Q6) {
            const uint8_t* src = W + (size_t)b * 208;
            lds_copy16_s(src, roff, raw);
            if (lane < 16) {
                lds_copy16_s(src + 192, rbase, raw + 1024);
                lds_copy4_s(W, rbase + (uint32_t)(nb * 208 + (b & ~1) * 2), raw + 1280);
            }
        } else {
            if constexpr (KP == 1) {
                if (lane < 48) lds_copy16_s(W, roff + (uint32_t)b * (g < 2 ? 128 : 16), raw);
            } else {
                lds_copy16_s(W + (size_t)b * 128, roff, raw);
                if (lane < 16) lds_copy16_s(W + (size_t)b * 16, rbase, raw + 1024);
            }
        }
        const uint8_t* src = rec + (size_t)b * 4 * REC;
#pragma unroll
        for (int i = 0; i < RECS / 1024; i++) lds_copy16_s(src + 1024 * i, 16 * lane, dst + 1024 * i);
        if (lane < RECS % 1024 / 16) lds_copy16_s(src + RECS / 1024 * 1024, 16 * lane, dst + RECS / 1024 * 1024);
    };
    static_assert(RECS % 1024 != 0, "copies per block");

    float accF[KP][KK][4], accM[KP][KK][4];
#pragma unroll
    for (int j = 0; j < KP; j++)
#pragma unroll
        for (int kk = 0; kk < KK; kk++)
#pragma unroll
            for (int i = 0; i < 4; i++) accF[j][kk][i] = accM[j][kk][i] = 0.0f;
    const NibMasks nm = nib_masks();
    Q6Masks m6{0x00f000f0u, 0x00300030u, 0x00c000c0u, 0x54005400u};
    asm("" : "+s"(m6.nib), "+s"(m6.lo2), "+s"(m6.hi2), "+v"(m6.exp));
    const h2v m1024 = {(_Float16)-1024.0f, (_Float16)-1024.0f}, m1152 = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    __syncthreads();  // the zero row
#pragma unroll
    for (int d = 0; d < kSmRing; d++) copy(d, L.ring[wave][d]);
    const f4v z = {0.0f, 0.0f, 0.0f, 0.0f};

    // one block; the lane's D registers are tokens t4 .. t4 + 3 of lane k
    auto block = [&](int b, SmSlot<PT, Q6, KP>& S) __attribute__((always_inline)) {
        wait_vmem_le<(kSmRing - 1) * kCopies>();
        asm volatile("" ::: "memory");
        const int odd = PT == 8 ? g >> 1 : 0, t4 = PT == 8 ? 4 * (g & 1) : 4 * g;
        // the records: A operands, lane (g, r) token r % PT of lane k, and
        // rows of PT floats: xs32 k, k + 4, xscale, xs16 x 4
        h8v av[KP][2];
        f4v xc[KP], xs[KP][KK], x0[KK], x8[KK];
#pragma unroll
        for (int j = 0; j < KP; j++) {
            const float* rf = (const float*)(S.rec[j] + PT * 128);
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const uint8_t* src = S.rec[j] + ((k * 4 + g) * PT + (c & (PT - 1))) * 16;
                if (PT == 8 && (c >> 3) != k) src = L.zero;
                av[j][k] = *(const h8v*)src;
            }
            xc[j] = *(const f4v*)&rf[2 * PT + t4];
#pragma unroll
            for (int kk = 0; kk < KK; kk++) {
                const int k = PT == 8 ? odd : kk;
                if constexpr (Q6) {
                    x0[kk] = *(const f4v*)&rf[(3 + k) * PT + t4];
                    x8[kk] = *(const f4v*)&rf[(5 + k) * PT + t4];
                } else {
                    xs[j][kk] = *(const f4v*)&rf[k * PT + t4];
                }
            }
        }
        if constexpr (Q6) {
            const Q6Raw& R = *(const Q6Raw*)S.raw;
            const int8_t* rsc = (const int8_t*)R.sc[c];
            float s0[KK], s8[KK];
#pragma unroll
            for (int kk = 0; kk < KK; kk++) {
                const int k = kp + 4 * (PT == 8 ? odd : kk);
                s0[kk] = (float)rsc[k];
                s8[kk] = (float)rsc[8 + k];
            }
            const uint32_t sv = *(const uint32_t*)&R.sc[c][4 * g] ^ 0x80808080u;
            const float d = factor_f16(R.dw[c] >> (16 * (b & 1)));
            uint2 ql[2];
            uint32_t qh[2];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                ql[k] = *(const uint2*)&R.q[16 * k + c][8 * (g >> 1)];
                qh[k] = *(const uint32_t*)&R.q[32 + 16 * k + c][8 * (kp & 1) + 4 * (g >> 1)];
            }
            f4v lo[KK], hi[KK];
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const h2v sc = __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, sv, k ? 0x04030401u : 0x04020400u)) + m1152;
                const h8v wl = q6_lows(ql[k], sc, g, m6), wh = q6_highs(qh[k], sc, g, m6);
                const int kk = KK == 1 ? 0 : k;
                lo[kk] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[0][k], wl, KK == 1 && k ? lo[kk] : z, 0, 0, 0);
                hi[kk] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[0][k], wh, KK == 1 && k ? hi[kk] : z, 0, 0, 0);
            }
            wait_lgkm0();
            copy(b + kSmRing, S);
#pragma unroll
            for (int kk = 0; kk < KK; kk++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float o2 = s0[kk] * (x0[kk][i] * 32.0f);             // VMULPS, ScaleF32(xs, 32)
                    o2 = fmaf(s8[kk], x8[kk][i] * 32.0f, o2);            // VFMADD231PS
                    accM[0][kk][i] = fmaf(d, o2, accM[0][kk][i]);
                    accF[0][kk][i] = fmaf(fmaf(hi[kk][i], 16.0f, lo[kk][i]), d * xc[0][i], accF[0][kk][i]);
                }
        } else {
            const uint8_t (*raw)[16] = (const uint8_t (*)[16])S.raw;
            const u4v h = *(const u4v*)raw[32 * KP + c];
            uint32_t nd[KP][2];
#pragma unroll
            for (int j = 0; j < KP; j++)
#pragma unroll
                for (int k = 0; k < 2; k++) nd[j][k] = *(const uint32_t*)&raw[32 * j + 16 * k + c][4 * g];
            const float d = f16_bits_to_f32(h.x & 0xffffu), dm = factor_f16(h.x >> 16);
            const uint32_t top = (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u);
            const uint32_t sb = ((g & 2) ? top : h.y & 0x3f3f3f3fu) >> (16 * (g & 1));
            const h2v one16 = {(_Float16)1.0f, (_Float16)0.0625f}, off16 = {(_Float16)-1024.0f, (_Float16)-64.0f};
            const h2v s = __builtin_elementwise_fma(
                __builtin_bit_cast(h2v, __builtin_amdgcn_perm(0x64646464u, sb, 0x04010400u)), one16, off16);
            const h2v n = s * m1024;
            f4v D[KP][KK];
#pragma unroll
            for (int j = 0; j < KP; j++) {
                D[j][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[j][0], dequant_nib(nd[j][0], s, n, nm), z, 0, 0, 0);
                D[j][KK - 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[j][1], dequant_nib(nd[j][1], s, n, nm),
                                                                      KK == 1 ? D[j][0] : z, 0, 0, 0);
            }
            wait_lgkm0();
            copy(b + kSmRing, S);
#pragma unroll
            for (int j = 0; j < KP; j++) {
                const int k8 = 8 * (kp + j);
                const float mlo = (float)__builtin_amdgcn_ubfe(h.z, k8, 6);
                const float mhi = (float)((__builtin_amdgcn_ubfe(h.z, k8 + 6, 2) << 4) | __builtin_amdgcn_ubfe(h.w, k8 + 4, 4));
#pragma unroll
                for (int kk = 0; kk < KK; kk++) {
                    const float mn = (PT == 8 ? odd : kk) ? mhi : mlo;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        accM[j][kk][i] = fmaf(dm, mn * xs[j][kk][i], accM[j][kk][i]);
                        accF[j][kk][i] = fmaf(D[j][kk][i], d * xc[j][i], accF[j][kk][i]);
                    }
                }
            }
        }
    };
#pragma unroll 1
    for (int b = 0; b < nb; b += kSmRing) {
#pragma unroll
        for (int d = 0; d < kSmRing; d++) {
            if (b + d >= nb) break;  // uniform
            block(b + d, L.ring[wave][d]);
        }
    }
    wait_vmem_le<0>();  // the last copies, never read
    // the reference's tree: s_kp = v_kp + v_(kp + 4), then (s0 + s1) + (s2 + s3)
#pragma unroll
    for (int j = 0; j < KP; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float v = accF[j][0][i] - accM[j][0][i];
            if constexpr (KK == 2) v = v + (accF[j][KK - 1][i] - accM[j][KK - 1][i]);
            L.ex[kp + j][lane][i] = v;
        }
    __syncthreads();
    for (int o = threadIdx.x; o < 16 * PT; o += 256 / KP) {
        const int t = o >> 4, r = o & 15;
        if (t >= job.p || row0 + r >= rows) continue;
        float s[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            s[q] = L.ex[q][16 * (t >> 2) + r][t & 3];
            if constexpr (KK == 1) s[q] = s[q] + L.ex[q][16 * (2 + (t >> 2)) + r][t & 3];
        }
        job.out[wi][(size_t)t * job.out_stride[wi] + row0 + r] = (s[0] + s[1]) + (s[2] + s[3]);
    }
}

// Batched Q4_K or Q6_K products of 2 to kTiledMinP rows (act.rec set); Q6_K
// blocks % 8 == 0; rows * rb < 4 GiB.
int launch_small_lanes(bool q6, SmallJob j, hipStream_t s) {
    if (j.n < 1 || j.n > 3 || !j.rec || j.p < 1 || j.p > kTiledMinP || j.blocks <= 0 || (q6 && j.blocks % 8))
        return fail(GLLM_EINVAL, "small batch: %d weights of %d blocks, %d tokens", j.n, j.blocks, j.p);
    int wg = 0;
    for (int i = 0; i < j.n; i++) {
        if (j.rows[i] <= 0 || (size_t)j.rows[i] * j.rb >= ((size_t)1 << 32))
            return fail(GLLM_EINVAL, "small batch: %d rows of %zu B", j.rows[i], j.rb);
        j.wg_begin[i] = wg;
        wg += (j.rows[i] + 15) / 16;
    }
    const dim3 grid(wg);
    const bool many = wg >= 2 * device_cus();
    if (q6 && j.p <= 8) hipLaunchKernelGGL((small_lanes_kernel<8, true, 1>), grid, dim3(256), 0, s, j);
    else if (q6) hipLaunchKernelGGL((small_lanes_kernel<16, true, 1>), grid, dim3(256), 0, s, j);
    else if (j.p <= 8 && many) hipLaunchKernelGGL((small_lanes_kernel<8, false, 2>), grid, dim3(128), 0, s, j);
    else if (j.p <= 8) hipLaunchKernelGGL((small_lanes_kernel<8, false, 1>), grid, dim3(256), 0, s, j);
    else hipLaunchKernelGGL((small_lanes_kernel<16, false, 1>), grid, dim3(256), 0, s, j);
    GLLM_HIP(hipGetLastError());
    return GLLM_OK;
}

// Q4_K from 8 rows on, after run_gemv's small batches (launch_small_lanes): 64 x
// 64 tiles split by AVX2 lane above 16 rows, which address a weight with 32-bit
// offsets, and 64 rows x 16 tokens (prefill_q4k_mfma_kernel) below.
int launch_q4k_mfma(const uint8_t* d_w, size_t rb, int rows, int blocks, const ActQ8& act, int p,
                    float* out, int out_stride, hipStream_t s) {
    if (rows <= 0 || blocks <= 0 || p <= 0) return GLLM_OK;
    PfArgs a{d_w, rb, rows, blocks, act, p, out, out_stride};
    const bool fits = (size_t)rows * rb < ((size_t)1 << 32);
    if (p > kTiledMinP) {
        if (!act.b16t || !fits)
            return fail(GLLM_EINVAL, "prefill: %d rows of %zu B need f16 tiles and < 4 GiB", rows, rb);
        GLLM_TRY(launch_q4k_lanes<false>(a, s));
    } else {
        launch_pf(a, s);  // 64-bit offsets
    }
    GLLM_HIP(hipGetLastError());
    return GLLM_OK;
}

}  // namespace gllm
