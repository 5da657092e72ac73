// gsd_prefill.hip -- the batched projection on 32 x 32 matrix-core tiles and
// the kernels between the projections of a prompt's layers (no reference
// kernel: the reference prefills token by token, run_gpu_native_chat.py:
// 1128-1130).
#include <algorithm>
#include <type_traits>

#include "gsd_device.h"
#include "gsd_internal.h"

// LDS addresses are formed as integers (an entry's address in one and-or, the
// base in the instruction's offset), and the LDS loads of lds_dma16 take theirs in m0
#pragma clang diagnostic ignored "-Wint-to-pointer-cast"
#pragma clang diagnostic ignored "-Winline-asm"

namespace gsd {
namespace {

typedef float float16v __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) const uint32_t lds_u32;
typedef __attribute__((address_space(3))) const u32x4v lds_u4;

// LDS byte address code * 128 + off (off < 128) of code j, a constant, of a
// lane's (aligned) word: 32 copies of an entry, one per lane of a half wave
template <bool B7>
__device__ __forceinline__ uint32_t code_addr32(const uint32_t (&w)[4], int j, uint32_t off) {
    if (B7) {
        const int s = 7 * j - 7, d = s >> 5;
        const uint32_t x = j == 0 ? w[0] << 7 : (d == 3 ? w[3] >> (s & 31) : __builtin_amdgcn_alignbit(w[d + 1], w[d], s & 31));
        return (x & 0x3F80u) | off;
    }
    const int b = j & 3;
    const uint32_t x = b == 0 ? w[j >> 2] << 7 : w[j >> 2] >> (8 * b - 7);
    return (x & 0x7F80u) | off;
}

// 64 lanes x 16 bytes from global memory into LDS at byte lds + 16 * lane,
// past the registers (no output register, so nothing is allocated to the
// load in flight; the caller waits on vmcnt before any wave reads the bytes).
// A scalar write of m0 needs one wait state before a load to LDS reads it, and
// the compiler adds none inside an asm block: without the s_nop the load could
// take the last m0 and put its 1 KB there.
__device__ __forceinline__ void lds_dma16(const void* p, uint32_t lds) {
    __asm__ volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(p) : "m0", "memory");
}

// y of one (token, row): the descaled sum s, kinks, rank-k
__device__ __forceinline__ float mm_finish(const MmSeg& w, const MmIn& in, int m, int row, float s) {
    float y = s * in.xs[m];
    if (w.row_ptr) {
        const uint32_t e = w.row_ptr[row + 1];
        for (uint32_t j = w.row_ptr[row]; j < e; j++) {
            const size_t at = (size_t)m * in.cols + w.kcols[j];
            y += w.kdel[j] * (in.Xf ? in.Xf[at] : __uint_as_float((uint32_t)in.X[at] << 16));
        }
    }
    for (int j = 0; j < w.k; j++) y += h2f(w.U[(size_t)row * w.k + j]) * w.tmp_k[(size_t)m * w.k + j];
    return y;
}

// ------------------------------------------------------------------------
// Batched projection, 32 x 32 x 16 matrix-core tiles.  Lattice form, packed
// tiles and operand fragments as hexmm_kernel: A = the tokens' (u, v) as
// fp16 (HL: high and low parts, two products per step), B = the rows'
// integer fields (r0, r1), exact, from the codebook in LDS; a 64-column
// block's sum is scaled by its fp16 scale into the fp32 accumulator.
//
// A block is NW waves, each 32 rows, over the same 32 T2 tokens, two blocks
// per CU.  Bound: the matrix cores (32 cycles per product) and, between them,
// the LDS: 16 code lookups and 8 T2 (high + low) or 4 T2 fragment reads per
// wave and stage, which follow each other and the products inside a wave.
// What the layout is for:
//  * 8 waves where there are rows for them: four waves per SIMD, of which some
//    read while others multiply, over the same LDS as two.  (4 waves of 64
//    rows read half the fragments but run two per SIMD: 44-48 % of the matrix
//    cores' cycles at 512 tokens, with either order of the reads, with raised
//    priorities, and with the memory's latency taken out.)  923-token prompt
//    3790 -> 3494 us, both on one card (others: 3584 to 3770);
//  * 32 x 32 tiles: one wave per SIMD issues 1.9 PFLOP/s of them and 1.1 of
//    16 x 16 tiles (fp16, measured alone), two waves 2.06 against 1.72;
//  * a lane's half of a 32-row tile comes from lanes (l & 15) + 32 (l >> 5)
//    and + 16 of the two 16-row tiles in memory, so neither the weights nor
//    the operands change their layout: step s = 2 q + t of a block takes
//    lane group 2 (l >> 5) + q and codes 4 t .. 4 t + 3;
//  * the tokens' fragments of a 64-column stage go from L2 straight into LDS,
//    three stages in turn, issued two ahead of the one that is read, with one
//    barrier per stage.  (The copies of the next chunk's codes and scales at a
//    chunk's end wait for all loads in the built loop: the first stage of a
//    chunk is issued two stages before that wait, the second one.)  Through
//    registers one stage ahead the latency of those loads took a third of the
//    time (high + low, 28672 x 4096, 512 tokens: 289 us, of which 118 went with
//    the fragment loads);
//  * 32 copies of the codebook (128 bytes per entry) instead of 64: the half
//    waves of a 4-byte LDS read are served in turn, and 28 KB for 217 points
//    leave room for two blocks per CU.
// Measured (MI355X, high + low operands, against 16 x 16 tiles with one
// block per CU): 4096 x 14336 at 512 tokens 143 -> 110 us (1.09 PFLOP/s of
// matrix-core work), 28672 x 4096 at 512 tokens 311 -> 260 us, at 37 tokens
// 64 -> 37 us, 6144 x 4096 (q, k and v) at 37 tokens 23 -> 17 us.
//
// Safety of the LDS stages.  Stage n goes to buffer n % 3 two stages ahead.
// A wave waits at least until only the younger loads than its share of stage n
// are in flight (vmcnt counts in issue order: the share of stage n + 1, NF loads,
// and in the second stage of a chunk the 3 code and scale loads issued
// after it) and for its own LDS reads, then meets the others; after that
// barrier all of stage n is in LDS and no wave reads stage n - 1, whose
// buffer stage n + 2 then overwrites.
// ------------------------------------------------------------------------
constexpr int kMmStages = 3;
template <int TB, bool HL, int T2, int NW>
__global__ void __launch_bounds__(NW * 64, NW / 2) hexmm32_kernel(const MmArgs a) {
    constexpr int TG = 2 * T2, RB = 2 * NW;   // 16-token groups and 16-row blocks of the block
    constexpr int NH = HL ? 2 : 1, FPS = 2 * NH;           // fragments of a token group and stage
    constexpr int NF = TG * FPS / NW;                      // fragments (1 KB) a wave moves per stage
    static_assert(NF >= 1 && TG * FPS % NW == 0, "every wave moves whole fragments");
    constexpr uint32_t ABYTES = TG * FPS * 1024, TBASE = kMmStages * ABYTES;
    static_assert(TBASE < 65536, "the codebook's base is an LDS instruction's offset");
    constexpr bool B7 = TB <= 128;
    constexpr int TBY = B7 ? kTile7 : kTileU8;
    extern __shared__ __attribute__((aligned(128))) unsigned char lds_mm[];   // stages, then the codebook
    const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nc = (a.in.cols + 127) >> 7, ng = (a.M + 15) >> 4, n_tt = (ng + TG - 1) / TG;
    const int sg = (a.nseg > 2 && (int)blockIdx.x >= a.seg[2].b0) ? 2 : (a.nseg > 1 && (int)blockIdx.x >= a.seg[1].b0) ? 1 : 0;
    const MmSeg& w = a.seg[sg];
    const int rows = w.rows, nrb = (rows + 15) >> 4, n_rt = (nrb + RB - 1) / RB;
    // the token tiles and column splits of one row tile on one XCD (blocks
    // go to the 8 XCDs in turn; b0 is a multiple of 8), the tensors' row tiles
    // dealt on from XCD to XCD
    const int S = w.nsplit, cps = (nc + S - 1) / S, bl = (int)blockIdx.x - w.b0;
    const int xcd = (bl + 8 - w.x0) & 7, bq = bl >> 3;
    const int rt = (bq / (n_tt * S)) * 8 + xcd, tt = (bq % (n_tt * S)) / S, ks = bq % S;
    if (rt >= n_rt) return;
    const int rb0 = rt * RB + wid * 2, g0 = tt * TG;
    const int c0 = ks * cps, c1 = min(nc, c0 + cps);
    if (c0 >= c1) return;
    const int half = (lane >> 4) & 1, kg = lane >> 5;
    const uint32_t sh7 = (uint32_t)(lane & 1) * 16u;

    // codes and scales of this wave's rows for chunk c
    const size_t ri = (size_t)min(rb0 + half, nrb - 1) * nc;
    const unsigned char* cp = reinterpret_cast<const unsigned char*>(w.codes_t) + ri * TBY + tile_lane_off(B7, (lane & 15) + 32 * kg);
    const uint32_t* sp = w.scales_t + ri * 16 + (lane & 15);
    constexpr int QOFF = B7 ? 28 * 8 : 16 * 16;   // from lane group 2 kg to 2 kg + 1 of a tile
    u32x4v cw[2];
    uint32_t sw;
    auto load = [&](int c) {
        c = min(c, nc - 1);
#pragma unroll
        for (int q = 0; q < 2; q++) cw[q] = *reinterpret_cast<const u32x4_a4*>(cp + (size_t)c * TBY + q * QOFF);
        sw = sp[(size_t)c * 16];
    };
    // this wave's fragments of stage 2 c + h (past the end: the last chunk's, unread)
    const u32x4v* ap[NF];
#pragma unroll
    for (int i = 0; i < NF; i++) {
        const int f = wid * NF + i, g = min(g0 + f / FPS, ng - 1), v = f % FPS;
        ap[i] = reinterpret_cast<const u32x4v*>(a.xa) + ((size_t)g * nc * (2 * FPS) + (HL ? (v >> 1) * 4 + (v & 1) : v)) * 64 + lane;
    }
    auto dma = [&](int st, uint32_t b) {
        const int c = min(st >> 1, nc - 1), h = st & 1;
#pragma unroll
        for (int i = 0; i < NF; i++) lds_dma16(ap[i] + ((size_t)c * (2 * FPS) + h * 2) * 64, b * ABYTES + (wid * NF + i) * 1024);
    };
    dma(2 * c0, 0);
    dma(2 * c0 + 1, 1);
    load(c0);
    for (int e = tid; e < TB * 32; e += NW * 64) reinterpret_cast<uint32_t*>(lds_mm + TBASE)[e] = a.fields[e >> 5];

    const uint32_t off = (uint32_t)(lane & 31) * 4u;
    const uint32_t aoff = (uint32_t)(half * FPS * 64 + (lane & 15) + 32 * kg) * 16u;
    uint32_t buf = 0;
    float16v acc[T2];
#pragma unroll
    for (int g = 0; g < T2; g++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[g][i] = 0.f;
    uint32_t w4[2][4], sc2;
    auto stage = [&](int c, auto hc) {
        constexpr int h = decltype(hc)::value;
        constexpr int NV = h ? NF + 3 : NF;   // loads younger than this wave's share of the stage
        __builtin_amdgcn_s_waitcnt((NV & 15) | ((NV >> 4) << 14) | 0x0F70);
        lds_barrier();
        const uint32_t Ab = buf * ABYTES + aoff;
        dma(2 * c + h + 2, buf == 0 ? 2 : buf - 1);
        buf = buf == 2 ? 0 : buf + 1;
        if constexpr (h == 0) {
            __builtin_amdgcn_sched_barrier(0);
            load(c + 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        half8v af[T2][4][NH], bw[4];
        auto frags = [&](int hl) {
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int g = 0; g < T2; g++)
                    af[g][s][hl] = __builtin_bit_cast(half8v, *(lds_u4*)(Ab + (2 * g * FPS + hl * 2 + (s & 1)) * 1024 + 256 * (s >> 1)));
        };
        frags(NH - 1);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            u32x4v b;
#pragma unroll
            for (int e = 0; e < 4; e++) b[e] = *(lds_u32*)(code_addr32<B7>(w4[s >> 1], 8 * h + 4 * (s & 1) + e, off) + TBASE);
            bw[s] = __builtin_bit_cast(half8v, b);
        }
        if constexpr (HL) frags(0);
        float16v d[T2];
#pragma unroll
        for (int g = 0; g < T2; g++)
#pragma unroll
            for (int i = 0; i < 16; i++) d[g][i] = 0.f;
        // (low parts first: the block's sum is rounded while it is small)
#pragma unroll
        for (int hl = NH - 1; hl >= 0; hl--)
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int g = 0; g < T2; g++) d[g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[g][s][hl], bw[s], d[g], 0, 0, 0);
        const float sc = h2f((uint16_t)(h ? (sc2 >> 16) : (sc2 & 0xFFFFu)));
#pragma unroll
        for (int g = 0; g < T2; g++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[g][i] = fmaf(d[g][i], sc, acc[g][i]);
    };
    for (int c = c0; c < c1; c++) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
#pragma unroll
            for (int i = 0; i < 4; i++) w4[q][i] = cw[q][i];
            if constexpr (B7) align7(w4[q], sh7);
        }
        sc2 = sw;
        stage(c, std::integral_constant<int, 0>{});
        stage(c, std::integral_constant<int, 1>{});
    }
    // (the two stages past the last chunk land before the block's LDS is
    // given back)
    __builtin_amdgcn_s_waitcnt(0x0F70);

    // lane: row l & 31 of the row tile, tokens 8 (i >> 2) + 4 kg + (i & 3)
    float* part = a.part + w.p0;
    const int Mp = ng * 16;
    const int row = rb0 * 16 + (lane & 31);
    if (row >= rows) return;
#pragma unroll
    for (int g = 0; g < T2; g++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int m = (g0 + 2 * g) * 16 + 8 * (i >> 2) + 4 * kg + (i & 3);
            if (m >= a.M) continue;
            if (S > 1) {   // this column split's sum; the consumer adds them in order
                part[((size_t)ks * Mp + m) * rows + row] = acc[g][i];
                continue;
            }
            const float y = mm_finish(w, a.in, m, row, acc[g][i]);
            float* yp = w.Y + (size_t)m * rows + row;
            *yp = a.accumulate ? *yp + y : y;
        }
}

// The partial sums of four consecutive rows of token m, in split order
__device__ __forceinline__ float4 part4(const float* part, const MmSeg& w, int Mp, int m, int row) {
    const float* p = part + w.p0 + (size_t)m * w.rows + row;
    const size_t st = (size_t)Mp * w.rows;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int k0 = 0; k0 < w.nsplit; k0 += 4) {
        float4 v[4];
#pragma unroll
        for (int k = 0; k < 4; k++)
            v[k] = k0 + k < w.nsplit ? *reinterpret_cast<const float4*>(p + (size_t)(k0 + k) * st) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            s.x += v[k].x;
            s.y += v[k].y;
            s.z += v[k].z;
            s.w += v[k].w;
        }
    }
    return s;
}
__device__ __forceinline__ float4 finish4(const float* part, const MmSeg& w, const MmIn& in, int Mp, int m, int row) {
    if (w.nsplit == 1) return *reinterpret_cast<const float4*>(w.Y + (size_t)m * w.rows + row);
    const float4 s = part4(part, w, Mp, m, row);
    return make_float4(mm_finish(w, in, m, row, s.x), mm_finish(w, in, m, row + 1, s.y), mm_finish(w, in, m, row + 2, s.z),
                       mm_finish(w, in, m, row + 3, s.w));
}

// Partial sums of a batched projection's tensors -> Y (one launch for all
// tensors: blockIdx.y)
__global__ void __launch_bounds__(256) mm_reduce_kernel(const MmArgs a) {
    const MmSeg& w = a.seg[blockIdx.y];
    if (w.nsplit == 1) return;
    const int r4 = w.rows >> 2, Mp = ((a.M + 15) >> 4) * 16;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < (size_t)a.M * r4; i += (size_t)gridDim.x * 256) {
        const int m = (int)(i / r4), row = (int)(i % r4) * 4;
        *reinterpret_cast<float4*>(w.Y + (size_t)m * w.rows + row) = finish4(a.part, w, a.in, Mp, m, row);
    }
}

// The token of a block of the two operand kernels, one block per token of ng
// groups of 16, or -1 (a block of the last round's groups past the end).  The
// 16 tokens of a group fill their lines of fragments 16 bytes each, so from 8
// groups on a group's blocks are on one XCD, whose L2 joins them (a 411-token
// chunk in block order wrote them from all 8: SwiGLU row of 14336 31 us
// against 26 for 512 tokens); fewer groups spread over the XCDs instead.
__device__ __forceinline__ int token_of_block(int ng) {
    const int b = (int)blockIdx.x;
    if (ng < 8) return b;
    const int j = b >> 3, g = (j >> 4) * 8 + (b & 7);
    return g < ng ? g * 16 + (j & 15) : -1;
}
dim3 token_grid(int M) {
    const int ng = (M + 15) / 16;
    return dim3(ng < 8 ? ng * 16 : (ng + 7) / 8 * 128);
}

// ------------------------------------------------------------------------
// Operands of the next projections from what the last launch left: the
// token's row (IN 0: X; 1: X plus the last projection, written back; 2:
// silu(gate) * up; 3: the embedding row of the token, written to X), RMSNorm
// where norm_w is given ((x * inv) * w, gsd_lq_cpu_engine.c:66-82), then its
// (u, v) as fp16 high and low parts after a per-token power of two, and the
// rank-k products of the tensors that read it.  One block per token (padded
// tokens of the last 16: zeros), the row in LDS; the last projection's column
// splits, descale, kinks and rank-k terms are taken in here, so a split
// projection needs no launch and no pass of its own.  Bound: memory (a
// 512-token chunk of the 7B shape reads and writes 25-60 MB).
// Measured (7B Precision, 512 tokens): in place of a partial-sum launch
// (13.5 us), a SwiGLU launch (15.8 us) and this pass reading their results
// (11-24 us).
// ------------------------------------------------------------------------
template <int IN, int NT>
__global__ void __launch_bounds__(NT) layer_prep_kernel(const LayerPrep p) {
    extern __shared__ __attribute__((aligned(16))) float xl[];   // the token's row
    __shared__ float red[NT / 64][2 * kMaxSeg + 2];
    constexpr float kS32 = 0.866025403784438646763723170752936183f;
    constexpr int NS = 2 * kMaxSeg;
    const int m = token_of_block((p.M + 15) >> 4);
    if (m < 0) return;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int cols = p.cols, nc = (cols + 127) >> 7, np = cols >> 1, nv4 = cols >> 2;
    const bool valid = m < p.M;
    float4* xl4 = reinterpret_cast<float4*>(xl);
    float4* X4 = reinterpret_cast<float4*>(p.X + (size_t)(valid ? m : 0) * cols);
    auto block_sums = [&](float (&v)[NS + 2], int n) {
        for (int s = 0; s < n; s++) {
            const float t = wave_sum_valu(v[s]);
            if (lane == 0) red[wid][s] = t;
        }
        __syncthreads();
        for (int s = 0; s < n; s++) {
            float t = 0.f;
            for (int q = 0; q < NT / 64; q++) t += red[q][s];
            v[s] = t;
        }
        __syncthreads();
    };
    const int Mp = ((p.M + 15) >> 4) * 16;
    const uint16_t* er = nullptr;
    if constexpr (IN == 3) er = p.embed + (size_t)p.tokens[valid ? m : 0] * cols;
    float ss = 0.f;
    for (int b = tid; b < nv4; b += NT) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (valid) {
            if constexpr (IN == 0) v = X4[b];
            if constexpr (IN == 1) {
                v = X4[b];
                const float4 y = finish4(p.part, p.last[0], p.in, Mp, m, 4 * b);
                v.x += y.x;
                v.y += y.y;
                v.z += y.z;
                v.w += y.w;
            }
            if constexpr (IN == 2) {
                const float4 g = finish4(p.part, p.last[0], p.in, Mp, m, 4 * b), u = finish4(p.part, p.last[1], p.in, Mp, m, 4 * b);
                v.x = g.x / (1.0f + expf(-g.x)) * u.x;
                v.y = g.y / (1.0f + expf(-g.y)) * u.y;
                v.z = g.z / (1.0f + expf(-g.z)) * u.z;
                v.w = g.w / (1.0f + expf(-g.w)) * u.w;
            }
            if constexpr (IN == 3) {
                const uint2 e = reinterpret_cast<const uint2*>(er)[b];
                v = make_float4(h2f((uint16_t)(e.x & 0xFFFFu)), h2f((uint16_t)(e.x >> 16)), h2f((uint16_t)(e.y & 0xFFFFu)),
                                h2f((uint16_t)(e.y >> 16)));
            }
            if constexpr (IN == 1 || IN == 3) {
                X4[b] = v;
                if (m == p.M - 1 && p.xlast) reinterpret_cast<float4*>(p.xlast)[b] = v;
            }
        }
        xl4[b] = v;
        ss = fmaf(v.x, v.x, ss);
        ss = fmaf(v.y, v.y, ss);
        ss = fmaf(v.z, v.z, ss);
        ss = fmaf(v.w, v.w, ss);
    }
    float sv[NS + 2];
    float inv = 1.f;
    if (p.norm_w) {
        sv[0] = ss;
        block_sums(sv, 1);
        inv = 1.0f / sqrtf(sv[0] / (float)cols + p.eps);
    }
    // x' in place (each thread its own float4s), its rank-k products and the
    // largest |u|, |v|
    const float4* w4 = reinterpret_cast<const float4*>(p.norm_w);
    const uint2* vt[NS];
    bool act[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        act[s] = (s & 1) < p.k[s >> 1];
        vt[s] = act[s] ? reinterpret_cast<const uint2*>(p.Vt[s >> 1] + (size_t)(s & 1) * cols) : nullptr;
        sv[s] = 0.f;
    }
    float mx = 0.f;
    for (int b = tid; b < nv4; b += NT) {
        float4 x = xl4[b];
        uint2 hv[NS];
#pragma unroll
        for (int s = 0; s < NS; s++) hv[s] = act[s] ? vt[s][b] : make_uint2(0u, 0u);
        if (p.norm_w) {
            const float4 nw = w4[b];
            x.x = (x.x * inv) * nw.x;
            x.y = (x.y * inv) * nw.y;
            x.z = (x.z * inv) * nw.z;
            x.w = (x.w * inv) * nw.w;
            xl4[b] = x;
        }
        if (valid && p.xn) reinterpret_cast<float4*>(p.xn + (size_t)m * cols)[b] = x;
        mx = fmaxf(mx, fmaxf(fabsf(x.x), fabsf(fmaf(kS32, x.y, 0.5f * x.x))));
        mx = fmaxf(mx, fmaxf(fabsf(x.z), fabsf(fmaf(kS32, x.w, 0.5f * x.z))));
#pragma unroll
        for (int s = 0; s < NS; s++) {
            if (!act[s]) continue;
            sv[s] = fmaf(x.x, h2f((uint16_t)(hv[s].x & 0xFFFFu)), sv[s]);
            sv[s] = fmaf(x.y, h2f((uint16_t)(hv[s].x >> 16)), sv[s]);
            sv[s] = fmaf(x.z, h2f((uint16_t)(hv[s].y & 0xFFFFu)), sv[s]);
            sv[s] = fmaf(x.w, h2f((uint16_t)(hv[s].y >> 16)), sv[s]);
        }
    }
    {
        const float t = wave_max_valu(mx);
        if (lane == 0) red[wid][NS] = t;
        block_sums(sv, act[0] || act[2] || act[4] ? NS : 0);   // (barriers in any case: x' and the maxima are in LDS)
        mx = red[0][NS];
        for (int q = 1; q < NT / 64; q++) mx = fmaxf(mx, red[q][NS]);
    }
#pragma unroll
    for (int s = 0; s < NS; s++)
        if (valid && tid == s && act[s]) p.tmp[s >> 1][(size_t)m * p.k[s >> 1] + (s & 1)] = sv[s] * p.S[s >> 1][s & 1];
    int ex = 0;
    if (mx > 0.f && mx < INFINITY) (void)frexpf(mx, &ex);
    const float up = ldexpf(1.f, 14 - ex);
    if (tid == 0) p.xs[m] = valid ? ldexpf(1.f, ex - 14) : 0.f;
    // fragments: four pairs (16 bytes) of the high parts and of the low parts per thread
    const int g16 = m >> 4, ml = m & 15;
    for (int i = tid; i < nc * 16; i += NT) {
        float4 f[2] = {make_float4(0.f, 0.f, 0.f, 0.f), make_float4(0.f, 0.f, 0.f, 0.f)};
        if (valid && 4 * i < np) {   // (np is a multiple of 32)
            f[0] = xl4[2 * i];
            f[1] = xl4[2 * i + 1];
        }
        const float xa[4] = {f[0].x, f[0].z, f[1].x, f[1].z}, xb[4] = {f[0].y, f[0].w, f[1].y, f[1].w};
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float u = xa[e] * up, v = fmaf(kS32, xb[e], 0.5f * xa[e]) * up;
            const _Float16 uh = (_Float16)u, vh = (_Float16)v;
            const _Float16 ul = (_Float16)(u - (float)uh), vl = (_Float16)(v - (float)vh);
            hi[e] = (uint32_t)__builtin_bit_cast(uint16_t, uh) | ((uint32_t)__builtin_bit_cast(uint16_t, vh) << 16);
            lo[e] = (uint32_t)__builtin_bit_cast(uint16_t, ul) | ((uint32_t)__builtin_bit_cast(uint16_t, vl) << 16);
        }
        const int q0 = 4 * i, c = q0 >> 6, h = (q0 >> 5) & 1, lg = (q0 >> 3) & 3, t2 = (q0 >> 2) & 1;
        uint4* o = p.xa + (((size_t)g16 * nc + c) * 8 + h * 2 + t2) * 64 + ml + 16 * lg;
        o[0] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        o[4 * 64] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    }
}

// ------------------------------------------------------------------------
// q, k, v of M prompt tokens: column splits, descale, kinks and rank-k terms
// taken in, then RoPE and the fp16 K/V append as rope_kv_kernel forms them
// (no contraction).  last[0] = q, [1] = k, [2] = v, or k and v only (nseg 2,
// the last layer's tokens before the last one).  A thread per pair.
// ------------------------------------------------------------------------
__global__ void __launch_bounds__(256) qkv_finish_kernel(const QkvFinish p) {
#pragma clang fp contract(off)
    const int half = p.r.hd >> 1, m = blockIdx.y, Mp = ((p.M + 15) >> 4) * 16;
    const int nq = p.nseg == 3 ? p.r.n_heads * half : 0, nk = p.r.n_kv * half;
    const int gid = blockIdx.x * 256 + threadIdx.x;
    if (gid >= nq + 2 * nk) return;
    const int which = gid < nq ? 0 : (gid < nq + nk ? 1 : 2);   // q, k, v
    const int pr = which == 0 ? gid : (which == 1 ? gid - nq : gid - nq - nk);
    const int s = p.nseg == 3 ? which : which - 1;
    const MmSeg& w = s == 0 ? p.last[0] : (s == 1 ? p.last[1] : p.last[2]);
    const int h = pr / half, i = pr % half;
    const bool pairs = p.r.interleaved || which == 2;   // (v: any two neighbours)
    const int i0 = h * p.r.hd + (pairs ? 2 * i : i), i1 = h * p.r.hd + (pairs ? 2 * i + 1 : i + half);
    float a, b;
    if (w.nsplit == 1) {
        a = w.Y[(size_t)m * w.rows + i0];
        b = w.Y[(size_t)m * w.rows + i1];
    } else {
        const float* pp = p.part + w.p0 + (size_t)m * w.rows;
        const size_t st = (size_t)Mp * w.rows;
        a = b = 0.f;
        for (int k = 0; k < w.nsplit; k++) {
            a += pp[k * st + i0];
            b += pp[k * st + i1];
        }
        a = mm_finish(w, p.in, m, i0, a);
        b = mm_finish(w, p.in, m, i1, b);
    }
    const int pos = p.r.pos + m;
    const size_t base = ((size_t)p.r.layer * p.r.max_seq + (size_t)pos) * (size_t)p.r.n_kv * p.r.hd;
    if (which == 2) {
        p.r.v_cache[base + i0] = f2h(a);
        p.r.v_cache[base + i1] = f2h(b);
        return;
    }
    const float2 cs = p.r.cs[(size_t)pos * half + i];
    const float x0 = a * cs.x - b * cs.y, x1 = a * cs.y + b * cs.x;
    if (which == 0) {
        float* q = p.q + (size_t)m * p.r.n_heads * p.r.hd;
        q[i0] = x0;
        q[i1] = x1;
    } else {
        p.r.k_cache[base + i0] = f2h(x0);
        p.r.k_cache[base + i1] = f2h(x1);
    }
}

// ------------------------------------------------------------------------
// Operands of bf16 tokens (single fp16 parts, as hexmm_xprep2_kernel) and
// the rank-k products of the tensors that read them, from one pass over X:
// one block per token (padded tokens: zeros), the row in registers.  A launch
// per tensor that read X again for its rank-k products took 7.7 us each at
// 128 tokens x 4096; this one takes 5 with two tensors' products.
// ------------------------------------------------------------------------
__global__ void __launch_bounds__(512) mm_xprep_kernel(const MmXprep p) {
    constexpr int NS = 2 * kMaxSeg;
    __shared__ float red[8][NS + 1];
    constexpr float kS32 = 0.866025403784438646763723170752936183f;
    const int m = token_of_block((p.M + 15) >> 4);
    if (m < 0) return;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int nc = (p.cols + 127) >> 7, ng8 = p.cols >> 3;
    const bool valid = m < p.M;
    const uint4* xr = reinterpret_cast<const uint4*>(p.X + (size_t)(valid ? m : 0) * p.cols);
    uint4 v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int i = tid + 512 * k;
        v[k] = valid && i < ng8 ? xr[i] : make_uint4(0u, 0u, 0u, 0u);
    }
    float sv[NS];
    bool act[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        act[s] = (s & 1) < p.k[s >> 1];
        sv[s] = 0.f;
    }
    float mx = 0.f;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int i = tid + 512 * k;
        const uint32_t w4[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
        float xa[4], xb[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            xa[e] = __uint_as_float(w4[e] << 16);
            xb[e] = __uint_as_float(w4[e] & 0xFFFF0000u);
            mx = fmaxf(mx, fmaxf(fabsf(xa[e]), fabsf(fmaf(kS32, xb[e], 0.5f * xa[e]))));
        }
#pragma unroll
        for (int s = 0; s < NS; s++) {
            if (!act[s] || i >= ng8) continue;
            const uint4 t = reinterpret_cast<const uint4*>(p.Vt[s >> 1] + (size_t)(s & 1) * p.cols)[i];
            const uint32_t t4[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                sv[s] = fmaf(xa[e], h2f((uint16_t)(t4[e] & 0xFFFFu)), sv[s]);
                sv[s] = fmaf(xb[e], h2f((uint16_t)(t4[e] >> 16)), sv[s]);
            }
        }
    }
    {
        const float t = wave_max_nonneg(mx);
        if (lane == 0) red[wid][NS] = t;
    }
#pragma unroll
    for (int s = 0; s < NS; s++) {
        if (!act[s]) continue;
        const float t = wave_sum_valu(sv[s]);
        if (lane == 0) red[wid][s] = t;
    }
    __syncthreads();
    mx = red[0][NS];
#pragma unroll
    for (int q = 1; q < 8; q++) mx = fmaxf(mx, red[q][NS]);
    if (valid && tid < NS && (tid & 1) < p.k[tid >> 1]) {
        float t = 0.f;
        for (int q = 0; q < 8; q++) t += red[q][tid];
        p.tmp[tid >> 1][(size_t)m * p.k[tid >> 1] + (tid & 1)] = t * p.S[tid >> 1][tid & 1];
    }
    int ex = 0;
    if (mx > 0.f && mx < INFINITY) (void)frexpf(mx, &ex);
    const float up = ldexpf(1.f, 14 - ex);
    if (tid == 0) p.xs[m] = valid ? ldexpf(1.f, ex - 14) : 0.f;
    const int g16 = m >> 4, ml = m & 15;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int i = tid + 512 * k;   // pairs 4 i .. 4 i + 3 (zeros past the row: chunk padding)
        if (i >= nc * 16) continue;
        const int q0 = 4 * i, c = q0 >> 6, h = (q0 >> 5) & 1, lg = (q0 >> 3) & 3, t2 = (q0 >> 2) & 1;
        const uint32_t w4[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
        uint32_t o[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float xa = __uint_as_float(w4[e] << 16), xb = __uint_as_float(w4[e] & 0xFFFF0000u);
            const float u = xa * up, vv = fmaf(kS32, xb, 0.5f * xa) * up;
            o[e] = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)u) | ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)vv) << 16);
        }
        p.xa[(((size_t)g16 * nc + c) * 4 + h * 2 + t2) * 64 + ml + 16 * lg] = make_uint4(o[0], o[1], o[2], o[3]);
    }
}

// ------------------------------------------------------------------------
// Causal attention of a batch of prompt tokens, head dims 64 and 128 (the
// arithmetic of attn_prefill_kernel, which keeps 256): token t of the batch
// at position p0 + t attends over cache positions 0 .. p0 + t.
// Block: KV head blockIdx.y and 64 query rows (T = 64 / G tokens x the G
// heads of the KV head), 8 waves: wave rt of a pair holds rows 32 rt .. + 31,
// one per lane column, and the four pairs take the 32-position chunks of the
// context in turn (c = pair, pair + 4, ..), each with LDS buffers of its own
// and one barrier per four chunks; their (max, sum, output) are merged in LDS
// at the end, in pair order.
// Bound: a wave's serial chain scores -> softmax -> output.  A block per 64
// rows fills 256 CUs with one wave per SIMD at 512 tokens, whose chain of 16 x
// 16 products took 2.2 us per 32 positions (107 us for 512 tokens behind 1024,
// 10 % of the matrix cores' rate; 32 us for 37 tokens behind 301, on 24 CUs).
// Splitting the context over pairs puts two waves on every SIMD and cuts the
// chain to a quarter; 32 x 32 products halve the LDS reads per row and leave
// a row's positions in two lanes; scores are masked only in chunks that reach
// past a row, and the output is rescaled only where a maximum moved.  Now 38
// us for the 512 tokens (0.56 PFLOP/s of matrix-core work).
// Scores: q as fp16 high + low parts after a per-row power of two (~22 bits),
// probabilities as high + low parts; K and V exact.  Positions past the
// block's last token are staged as zeros (cache rows there may hold anything).
// ------------------------------------------------------------------------
template <int HD>
__global__ void __launch_bounds__(512, 2) attn_prompt_kernel(const PrefillAttn a) {
    constexpr int NP = 4;         // pairs of waves
    constexpr int KS = HD + 8;    // K row stride, halves (16 bytes of padding)
    constexpr int VS = 36;        // V^T row stride, halves (32 positions + 4)
    constexpr int NKS = HD / 16;  // steps of the scores
    constexpr int NDT = HD / 32;  // 32-dimension tiles of the output
    constexpr int D8 = HD / 8;    // 16-byte pieces of a cache row
    constexpr int NK = 32 * D8 / 128, NV = 16 * D8 / 128;   // K pieces, V pairs of pieces per thread and chunk
    constexpr uint32_t KB = 32 * KS * 2, BUF = KB + HD * VS * 2;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_pa[];   // [pair][2][K rows | V^T rows], then the merge
    const int tid = threadIdx.x, lane = tid & 63, gt = tid & 127;
    const int pair = __builtin_amdgcn_readfirstlane(tid >> 7), rt = __builtin_amdgcn_readfirstlane((tid >> 6) & 1);
    const int n = lane & 31, kg = lane >> 5;
    const int lg = a.log2g, G = 1 << lg, T = 64 >> lg;
    const int grp = (int)gridDim.x - 1 - (int)blockIdx.x;   // the longest blocks first
    const int kvh = (int)blockIdx.y, t0 = grp * T;
    const int r = 32 * rt + n;
    const int t = t0 + (r >> lg), head = kvh * G + (r & (G - 1));
    const bool valid = t < a.M;
    const int limit = a.p0 + t;   // last position of this row
    const int maxpos = a.p0 + min(t0 + T, a.M) - 1;
    const int nch = maxpos / 32 + 1, nround = (nch + NP - 1) / NP;
    const int full = (a.p0 + t0 + ((32 * rt) >> lg) + 1) / 32;   // chunks below every row of this wave

    half8v qh[NKS], ql[NKS];   // B: row n, dims 16 ks + 8 kg ..
    float down;
    {
        const float qs = a.sm_scale * 1.44269504088896340736f;
        const float* qr = a.q + ((size_t)(valid ? t : 0) * a.n_heads + head) * HD + 8 * kg;
        float qv[NKS][8];
        float mx = 0.f;
#pragma unroll
        for (int ks = 0; ks < NKS; ks++) {
            float4 f0 = make_float4(0.f, 0.f, 0.f, 0.f), f1 = f0;
            if (valid) {
                f0 = *reinterpret_cast<const float4*>(qr + 16 * ks);
                f1 = *reinterpret_cast<const float4*>(qr + 16 * ks + 4);
            }
            const float v8[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
#pragma unroll
            for (int j = 0; j < 8; j++) {
                qv[ks][j] = v8[j] * qs;
                mx = fmaxf(mx, fabsf(qv[ks][j]));
            }
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        int ex = 0;
        if (mx > 0.f && mx < INFINITY) (void)frexpf(mx, &ex);
        const float up = ldexpf(1.f, 14 - ex);
        down = ldexpf(1.f, ex - 14);
#pragma unroll
        for (int ks = 0; ks < NKS; ks++)
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float x = qv[ks][j] * up;
                const _Float16 h = (_Float16)x;
                qh[ks][j] = h;
                ql[ks][j] = (_Float16)(x - (float)h);
            }
    }

    const size_t rstride = (size_t)a.n_kv * HD;   // halves from one position to the next
    const size_t lbase = ((size_t)a.layer * a.max_seq * a.n_kv + kvh) * HD;
    const uint16_t* kbase = a.k_cache + lbase;
    const uint16_t* vbase = a.v_cache + lbase;
    u32x4v kr[NK], vr[NV][2];
    const u32x4v z4 = {0u, 0u, 0u, 0u};
    auto fetch = [&](int c) {
#pragma unroll
        for (int i = 0; i < NK; i++) {
            const int idx = gt + 128 * i, p = 32 * c + idx / D8;
            kr[i] = p <= maxpos ? *reinterpret_cast<const u32x4v*>(kbase + (size_t)p * rstride + (idx % D8) * 8) : z4;
        }
#pragma unroll
        for (int i = 0; i < NV; i++) {   // pairs of positions (low bits) x pieces
            const int idx = gt + 128 * i, p = 32 * c + 2 * (idx & 15);
            const size_t off = (size_t)p * rstride + (idx >> 4) * 8;
            vr[i][0] = p <= maxpos ? *reinterpret_cast<const u32x4v*>(vbase + off) : z4;
            vr[i][1] = p + 1 <= maxpos ? *reinterpret_cast<const u32x4v*>(vbase + off + rstride) : z4;
        }
    };
    unsigned char* const mine = lds_pa + (uint32_t)pair * 2u * BUF;
    auto put = [&](int b) {
        uint16_t* kl = reinterpret_cast<uint16_t*>(mine + b * BUF);
        uint32_t* vw = reinterpret_cast<uint32_t*>(mine + b * BUF + KB);
#pragma unroll
        for (int i = 0; i < NK; i++) {
            const int idx = gt + 128 * i;
            *reinterpret_cast<u32x4v*>(kl + (idx / D8) * KS + (idx % D8) * 8) = kr[i];
        }
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int idx = gt + 128 * i, j = idx & 15, d0 = (idx >> 4) * 8;
#pragma unroll
            for (int e = 0; e < 8; e++)   // dim d0 + e of positions 2 j, 2 j + 1
                vw[(d0 + e) * (VS / 2) + j] = __builtin_amdgcn_perm(vr[i][1][e >> 1], vr[i][0][e >> 1], e & 1 ? 0x07060302u : 0x05040100u);
        }
    };

    float16v o[NDT];
#pragma unroll
    for (int d = 0; d < NDT; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[d][i] = 0.f;
    float mrun = -INFINITY, lsum = 0.f;
    if (pair < nch) {
        fetch(pair);
        put(0);
    }
    __syncthreads();
    for (int i = 0; i < nround; i++) {
        const int c = pair + NP * i;
        if (c + NP < nch) fetch(c + NP);
        if (c < nch) {
            const uint16_t* kb = reinterpret_cast<const uint16_t*>(mine + (i & 1) * BUF);
            const uint16_t* vb = reinterpret_cast<const uint16_t*>(mine + (i & 1) * BUF + KB);
            float16v sh, sl;
#pragma unroll
            for (int j = 0; j < 16; j++) sh[j] = sl[j] = 0.f;
#pragma unroll
            for (int ks = 0; ks < NKS; ks++) {
                const half8v ka = *reinterpret_cast<const half8v*>(kb + n * KS + 16 * ks + 8 * kg);
                sh = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka, qh[ks], sh, 0, 0, 0);
                sl = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka, ql[ks], sl, 0, 0, 0);
            }
            // lane: row n, positions 32 c + 8 (j >> 2) + 4 kg + (j & 3)
            float s[16];
#pragma unroll
            for (int j = 0; j < 16; j++) s[j] = (sh[j] + sl[j]) * down;
            if (c >= full) {
#pragma unroll
                for (int j = 0; j < 16; j++)
                    if (32 * c + 8 * (j >> 2) + 4 * kg + (j & 3) > limit) s[j] = -INFINITY;
            }
            float mc = s[0];
#pragma unroll
            for (int j = 1; j < 16; j++) mc = fmaxf(mc, s[j]);
            mc = fmaxf(mc, __shfl_xor(mc, 32, 64));
            const float mnew = fmaxf(mrun, mc);
            const float base = mnew == -INFINITY ? 0.f : mnew;   // (a chunk past this row: all masked)
            if (__any(mnew != mrun)) {
                const float alpha = __builtin_amdgcn_exp2f(mrun - base);
                lsum *= alpha;
#pragma unroll
                for (int d = 0; d < NDT; d++)
#pragma unroll
                    for (int j = 0; j < 16; j++) o[d][j] *= alpha;
                mrun = mnew;
            }
            half8v ph[2], pl[2];
#pragma unroll
            for (int j = 0; j < 16; j++) {
                const float pj = __builtin_amdgcn_exp2f(s[j] - base);
                lsum += pj;
                const _Float16 h = (_Float16)pj;
                ph[j >> 3][j & 7] = h;
                pl[j >> 3][j & 7] = (_Float16)(pj - (float)h);
            }
#pragma unroll
            for (int st = 0; st < 2; st++) {
#pragma unroll
                for (int d = 0; d < NDT; d++) {   // A: dim 32 d + n, positions 16 st + 4 kg .. + 3 and 8 on
                    const uint16_t* vrow = vb + (32 * d + n) * VS + 16 * st + 4 * kg;
                    const uint2 lo4 = *reinterpret_cast<const uint2*>(vrow), hi4 = *reinterpret_cast<const uint2*>(vrow + 8);
                    const u32x4v vw = {lo4.x, lo4.y, hi4.x, hi4.y};
                    const half8v va = __builtin_bit_cast(half8v, vw);
                    o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, pl[st], o[d], 0, 0, 0);
                    o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, ph[st], o[d], 0, 0, 0);
                }
            }
        }
        if (c + NP < nch) put((i + 1) & 1);
        __syncthreads();
    }
    lsum += __shfl_xor(lsum, 32, 64);

    // merge the pairs: maxima and sums, then the scaled outputs, dim tile d
    // of a row tile summed and stored by its pair d
    float2* ml = reinterpret_cast<float2*>(lds_pa);          // [rt][pair][32 rows]
    float4* ob = reinterpret_cast<float4*>(lds_pa + 2048);   // [rt][pair][tile][4][64 lanes]
    if (kg == 0) ml[(rt * NP + pair) * 32 + n] = make_float2(mrun, lsum);
    __syncthreads();
    float M = -INFINITY, L = 0.f;
#pragma unroll
    for (int p = 0; p < NP; p++) M = fmaxf(M, ml[(rt * NP + p) * 32 + n].x);
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const float2 v = ml[(rt * NP + p) * 32 + n];
        L += v.y * __builtin_amdgcn_exp2f(v.x - M);
    }
    const float f = __builtin_amdgcn_exp2f(mrun - M);
#pragma unroll
    for (int d = 0; d < NDT; d++)
#pragma unroll
        for (int j = 0; j < 4; j++)
            ob[(((rt * NP + pair) * NDT + d) * 4 + j) * 64 + lane] =
                make_float4(o[d][4 * j] * f, o[d][4 * j + 1] * f, o[d][4 * j + 2] * f, o[d][4 * j + 3] * f);
    __syncthreads();
    if (pair < NDT && valid) {
        const float inv = 1.0f / L;
        float* out = a.out + ((size_t)t * a.n_heads + head) * HD + 32 * pair + 4 * kg;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float4 y = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int p = 0; p < NP; p++) {
                const float4 v = ob[(((rt * NP + p) * NDT + pair) * 4 + j) * 64 + lane];
                y.x += v.x;
                y.y += v.y;
                y.z += v.z;
                y.w += v.w;
            }
            *reinterpret_cast<float4*>(out + 8 * j) = make_float4(y.x * inv, y.y * inv, y.z * inv, y.w * inv);
        }
    }
}

template <int HD>
hipError_t launch_attn_prompt_t(const PrefillAttn& a, dim3 grid, hipStream_t st) {
    constexpr int lds = 4 * 2 * (32 * (HD + 8) * 2 + HD * 36 * 2);
    static_assert(lds >= 2048 + 2 * 4 * (HD / 32) * 4 * 64 * 16 && lds <= 160 * 1024, "the merge fits the stages");
    static LdsLimit limit;
    const hipError_t e = raise_lds_limit(limit, reinterpret_cast<const void*>(&attn_prompt_kernel<HD>), lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((attn_prompt_kernel<HD>), grid, dim3(512), lds, st, a);
    return hipGetLastError();
}

template <int TB, bool HL, int T2, int NW>
hipError_t launch_hexmm32_t(const MmArgs& a, int grid, hipStream_t st) {
    const int lds = kMmStages * 2 * T2 * (HL ? 4 : 2) * 1024 + TB * 128;
    static LdsLimit limit;
    const hipError_t e = raise_lds_limit(limit, reinterpret_cast<const void*>(&hexmm32_kernel<TB, HL, T2, NW>), lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((hexmm32_kernel<TB, HL, T2, NW>), dim3(grid), dim3(NW * 64), lds, st, a);
    return hipGetLastError();
}

template <int TB>
hipError_t launch_hexmm32_tb(const MmArgs& a, int grid, hipStream_t st) {
    if (a.hl) {
        if (a.nw == 8 && a.t2 == 2) return launch_hexmm32_t<TB, true, 2, 8>(a, grid, st);
        if (a.nw == 4 && a.t2 == 1) return launch_hexmm32_t<TB, true, 1, 4>(a, grid, st);
        return hipErrorInvalidValue;
    }
    if (a.nw == 8 && a.t2 == 2) return launch_hexmm32_t<TB, false, 2, 8>(a, grid, st);
    if (a.nw == 4 && a.t2 == 4) return launch_hexmm32_t<TB, false, 4, 4>(a, grid, st);
    if (a.nw == 4 && a.t2 == 2) return launch_hexmm32_t<TB, false, 2, 4>(a, grid, st);
    if (a.nw == 4 && a.t2 == 1) return launch_hexmm32_t<TB, false, 1, 4>(a, grid, st);
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_attn_prompt(const PrefillAttn& a, dim3 grid, hipStream_t st) {
    if (a.hd == 64) return launch_attn_prompt_t<64>(a, grid, st);
    if (a.hd == 128) return launch_attn_prompt_t<128>(a, grid, st);
    return hipErrorInvalidValue;
}

bool hexmm32_codebook(int n_pts) { return n_pts == 217 || n_pts == 127; }

// High + low operands (a prompt): 8 waves over 64 tokens from 33 tokens on (37
// tokens, 28672 x 4096: 37 us against 41 with 4 waves), 4 over 32 below, where
// the grid is finer and less of a tile is padding.  The columns are split into
// what fills two blocks per CU (at least 4 chunks each; up to 16, whose
// partial sums the next launch still takes in within its own time).
MmTile hexmm32_tile_hl(int M, int rows_total_tiles_of_16, int cols) {
    const int ng = (M + 15) / 16, nc = (cols + 127) / 128, ncu = device_cu_count() > 0 ? device_cu_count() : 256;
    MmTile t{ng <= 2 ? 4 : 8, ng <= 2 ? 1 : 2, 1};
    const int rb = 2 * t.nw, tiles = ((rows_total_tiles_of_16 + rb - 1) / rb) * ((ng + 2 * t.t2 - 1) / (2 * t.t2));
    t.nsplit = whole_splits(nc, std::max(1, std::min({2 * ncu / tiles, nc / 4, 16})));
    return t;
}

// Single operands (gsdh_model_matmul), one tensor of a call (tensors of one
// call tile alike, so a launch may hold several): 4 waves over 32 or 64 tokens,
// from 65 on over 128, which decode a weight least often, or 8 waves over 64
// where tiles of 128 would hold more padding (with the passes, 8 waves against
// 4: 28672 x 4096 at 300 tokens 155 and 175 us, 4096 x 14336 96 and 105; at 512
// 234 and 245, 124 and 122; at 128 92 and 93, 68 and 70).  nsplit 0: hexmm_kernel, where the columns would have to be
// split and the partial sums' passes (8 bytes per split and output) come to
// more than about the decode of the weights they spare: measured at 512
// tokens 4096 x 4096, 37 us there against 31 + 13 here; 4096 x 14336 in four
// splits 110 against 75 + 13; 28672 x 4096 at 128 tokens in two 57 against
// 48 + 8, 6144 x 4096 at 16 tokens 13 + 4 (three launches of each) against 9 + 3.
MmTile hexmm32_tile(int M, int rows, int cols) {
    const int ng = (M + 15) / 16, nc = (cols + 127) / 128, ncu = device_cu_count() > 0 ? device_cu_count() : 256;
    const bool t128 = ng > 4 && (ng + 7) / 8 * 2 == (ng + 3) / 4;
    MmTile t{ng <= 4 || t128 ? 4 : 8, ng <= 2 ? 1 : (t128 ? 4 : 2), 0};
    const int tiles = ((rows + 32 * t.nw - 1) / (32 * t.nw)) * ((ng + 2 * t.t2 - 1) / (2 * t.t2));
    const int s = whole_splits(nc, std::max(1, std::min({(nc >= 64 ? 2 * ncu : ncu) / tiles, nc / 4, 16})));
    const bool ok = ng <= 4 || (s == 1 ? 4 * tiles >= 3 * ncu : 32LL * s * ng * 16 <= 5LL * cols);
    t.nsplit = ok && rows % 4 == 0 ? s : 0;
    return t;
}

// Fills seg[].b0, .x0, .nsplit and .p0 for the tile; returns the floats of partial
// sums (seg[].rows set).  Tensors of one launch that are split differently
// keep their own split (nsplit 0: the tile's).  A tensor's row tiles begin on
// the XCD after the last tensor's end: with every tensor's from XCD 0 on, the
// four row tiles each of k and v (7B shape, 512 tokens) kept four XCDs busy
// while the others waited (q, k, v: 70 us against 49; k and v alone 50, 29).
size_t hexmm32_layout(MmArgs& a, const MmTile& t, int* grid) {
    const int ng = (a.M + 15) / 16, n_tt = (ng + 2 * t.t2 - 1) / (2 * t.t2);
    int b = 0, x = 0;
    size_t p = 0;
    a.nw = t.nw;
    a.t2 = t.t2;
    for (int s = 0; s < a.nseg; s++) {
        MmSeg& w = a.seg[s];
        if (w.nsplit <= 0) w.nsplit = t.nsplit;
        const int n_rt = ((w.rows + 15) / 16 + 2 * t.nw - 1) / (2 * t.nw);
        w.b0 = b;
        w.x0 = x;
        w.p0 = p;
        b += 8 * n_tt * w.nsplit * ((n_rt + 7) / 8);
        x = (x + n_rt) & 7;
        if (w.nsplit > 1) p += (size_t)w.nsplit * ng * 16 * w.rows;
    }
    *grid = b;
    return p;
}

hipError_t launch_hexmm32(const MmArgs& a, int grid, hipStream_t st) {
    if (a.M <= 0 || a.in.cols <= 0 || a.in.cols % 64 || a.nseg < 1 || a.nseg > kMaxSeg || !a.xa || !a.in.xs || !a.fields)
        return hipErrorInvalidValue;
    for (int s = 0; s < a.nseg; s++) {
        const MmSeg& w = a.seg[s];
        if (!w.codes_t || !w.scales_t || w.rows <= 0 || w.nsplit < 1 || (w.nsplit > 1 && !a.part) || (w.nsplit == 1 && !w.Y) ||
            (w.k > 0 && (!w.U || !w.tmp_k)) || (w.row_ptr && !a.in.Xf && !a.in.X))
            return hipErrorInvalidValue;
    }
    if (a.n_pts == 217) return launch_hexmm32_tb<217>(a, grid, st);
    if (a.n_pts == 127) return launch_hexmm32_tb<127>(a, grid, st);
    return hipErrorInvalidValue;
}

hipError_t launch_mm_reduce(const MmArgs& a, hipStream_t st) {
    size_t n = 0;
    for (int s = 0; s < a.nseg; s++) {
        if (a.seg[s].nsplit == 1) continue;
        if (a.seg[s].rows % 4) return hipErrorInvalidValue;
        n = std::max(n, (size_t)a.M * (a.seg[s].rows / 4));
    }
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(mm_reduce_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 4096), a.nseg), dim3(256), 0, st, a);
    return hipGetLastError();
}

bool mm_xprep_covers(const MmXprep& p) {
    if (p.cols > 16384 || (reinterpret_cast<uintptr_t>(p.X) & 15)) return false;
    for (int s = 0; s < kMaxSeg; s++)
        if (p.k[s] > 2 || (p.k[s] > 0 && (reinterpret_cast<uintptr_t>(p.Vt[s]) & 15))) return false;
    return true;
}

hipError_t launch_mm_xprep(const MmXprep& p, hipStream_t st) {
    if (p.M <= 0 || p.cols <= 0 || p.cols % 64 || !p.X || !p.xa || !p.xs || !mm_xprep_covers(p)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(mm_xprep_kernel, token_grid(p.M), dim3(512), 0, st, p);
    return hipGetLastError();
}

hipError_t launch_layer_prep(const LayerPrep& p, LayerPrepIn in, hipStream_t st) {
    if (p.M <= 0 || p.cols <= 0 || p.cols % 64 || p.cols > kLayerPrepMaxCols || !p.xa || !p.xs) return hipErrorInvalidValue;
    const size_t lds = (size_t)p.cols * 4;
    const dim3 grid = token_grid(p.M);
    // up to a block per CU: 16 waves each, for the loads in flight (37 tokens,
    // SwiGLU row of 14336: 20.4 -> 15.0 us); more blocks share the CUs and
    // are faster with 8 (512 tokens: 26.8 against 30.6, 304: 24.1 both)
    const bool wide = (int)grid.x <= (device_cu_count() > 0 ? device_cu_count() : 256);
#define GSD_PREP_N(IN, NT)                                                                                               \
    {                                                                                                                    \
        static LdsLimit limit;                                                                                           \
        const hipError_t e = raise_lds_limit(limit, reinterpret_cast<const void*>(&layer_prep_kernel<IN, NT>), lds);     \
        if (e != hipSuccess) return e;                                                                                   \
        hipLaunchKernelGGL((layer_prep_kernel<IN, NT>), grid, dim3(NT), lds, st, p);                                     \
    }
#define GSD_PREP(IN) if (wide) GSD_PREP_N(IN, 1024) else GSD_PREP_N(IN, 512) break;
    switch (in) {
        case kPrepRow: GSD_PREP(0)
        case kPrepResidual: GSD_PREP(1)
        case kPrepSwiGLU: GSD_PREP(2)
        case kPrepEmbed: GSD_PREP(3)
    }
#undef GSD_PREP
#undef GSD_PREP_N
    return hipGetLastError();
}

hipError_t launch_qkv_finish(const QkvFinish& p, hipStream_t st) {
    if (p.M <= 0 || (p.nseg != 2 && p.nseg != 3) || !p.r.cs || p.r.pos < 0 || p.r.pos + p.M > p.r.max_seq) return hipErrorInvalidValue;
    const int half = p.r.hd / 2, n = (p.nseg == 3 ? p.r.n_heads * half : 0) + 2 * p.r.n_kv * half;
    hipLaunchKernelGGL(qkv_finish_kernel, dim3((n + 255) / 256, p.M), dim3(256), 0, st, p);
    return hipGetLastError();
}

}  // namespace gsd
