// Fused chunked-SSD prefill in fp32 for d_state 128 / headdim 64 / rank 2 (the d_model 768
// KulaMamba in fp32), gfx950.
//
// Same algorithm and formulation as the bf16 MFMA kernel (m3_ssd_mfma.hip): the quadratic
// form inside a chunk and the state carried across chunks (mamba3/ssd.py:118-244), with the
// layer's preparation fused (mamba3/mamba3.py:197-256), the trapezoid folded into
// a_u = lambda_u dt_u and b_u = (1 - lambda_{u+1}) dt_{u+1} so the contraction rank stays R.
// Every operand stays fp32: the contractions run on v_mfma_f32_16x16x4_f32 (lane l supplies
// A[l%16][l/16] and B[l/16][l%16]; it holds D[4(l/16)+v][l%16]).
//
// Launches:
//   1. bc_norm_f32: per (token, group), B^ = RMSNorm(B) * w + bias and C^ likewise, fp32, in
//      the reference's (n, r) order (mamba3/mamba3.py:19-35, 147-157).
//   2. for sequences of more than two segments, ssd_f32<false>: a state-only walk of every
//      segment of the sequence but the last, from a zero state in its own RoPE frame, and
//      seg_combine_f32, which turns the end states into the states entering each segment;
//   3. ssd_f32<true>: one 768-thread workgroup per (batch, head, segment) walks its chunks of
//      Q = 32 tokens (64 rows (t, r) = 2t + r).
//
// Waves 0-3 are column waves: each carries its 16 headdim columns of the fp32 state H^T [n][p]
// in MFMA accumulators and computes their outputs. Waves 4-11 are helpers: they compute the
// scores and prepare the next chunk's tiles. Per chunk, two phases with a barrier after each:
//   scores    column waves  G3  Y = diag(e^{c_t}) C~ H^T (H^T straight from the accumulators:
//                               accumulator v of lane group g is row n = 16 t + 4 g + v, the
//                               contraction slot of MFMA step v, whose C~ operands are one
//                               128-bit read for four steps)
//             helpers       X^T; G1  S = (C~ B~^T) * Lc on the 10 causal 16 x 16 blocks,
//                               Lc[t][u] = [u<=t] exp(c_t - c_u) (a_u + [u<t] b_u), D on the diagonal;
//                           the next chunk's angle sums, the token scalars of the one after it
//   update    column waves  G2  Y += S X, out = sum_r mimo_down_r silu(z mimo_z_r) y_r
//                               (mamba3/mamba3.py:233-239)
//                           G4  H^T = e^{c_end} H^T + B~^T (diag(w) X), w_u = e^{c_end - c_u} (a_u + b_u)
//             helpers       angles and rotated C~ / B~ tiles (mamba3/mamba3.py:38-45, 160-166) of
//                           the next chunk
// B~ is kept twice (G4 reads it while the helpers write the next chunk's), which balances the
// phases: 208-224 MFMAs per SIMD in the first, 168 in the second.
// For the training forward (M3_FLAG_FOR_BACKWARD) the walk also stores, from the values it
// holds, the per-token operands the layer backward reads, in the staged fp32 layer path's
// layouts (m3_layer_fp32.hip), and its chunk-start states.
//
// Bound by SIMD issue: 1,504 v_mfma_f32_16x16x4_f32 of 32 cycles per chunk are 12.0K cycles on
// four SIMDs, 5,000 other VALU instructions 5.0K, and they add up, with 2.7K of waits at the two
// barriers, to 19.7K, 8.2 us per chunk and workgroup (profiles/pmc_segmented_prefill_kernels.md).
// d_model 768 over 4 x 1024 tokens (96 (batch, head) pairs), from a cool clock: 300 us with two
// workgroups of 32 columns per pair, state and operands through LDS, all eight waves in step;
// 212 us with this split (135 + 70 state pass + 7); 193 at the sustained clock (118 + 62 + 7 and
// the normalisation).
#include <algorithm>

#include "m3_common.h"
#include "m3_kernels.h"
#include "m3_mfma.h"
#include "m3_segments.h"

namespace m3 {
namespace f32k {

constexpr int Q = 32;
constexpr int N = 128;
constexpr int P = 64;
constexpr int R = 2;
constexpr int NR = N * R;
constexpr int NH = N / 2;
constexpr int ROWS = Q * R;
constexpr int CW = 4, HW = 8;         // column and helper waves
constexpr int HT = 64 * HW;
constexpr int THREADS = 64 * (CW + HW);
constexpr int LPT = N / 4;            // helper lanes per token: two RoPE pairs each
constexpr int GR = HT / LPT;          // token groups of a chunk
constexpr int TPT = Q / GR;           // tokens per group
constexpr int XTOK = Q * P / HT;      // X elements per helper thread: consecutive tokens of one column
constexpr int NT = N / 16;            // state row tiles
// LDS row strides of 4 (mod 64) words: the 128-bit operand reads of 16 rows and the 32-bit
// reads of 16 columns in rows 4 apart (G4) each touch every bank once.
constexpr int CST = N + 4;
constexpr int SST = ROWS + 4;

struct Tok {
    float c[Q];   // inclusive prefix of A dt over the chunk
    float ec[Q];  // exp(c_t)
    float av[Q], bv[Q];  // a_u = lambda_u dt_u, b_u = (1 - lambda_{u+1}) dt_{u+1}
    float w[Q];   // exp(c_end - c_u) (a_u + b_u)
    float dt[Q], lam[Q];
    float sb[Q];  // (1 - lambda_{u+1}) exp(A dt_{u+1}): x_b of the next token over x_r of this one
    float cend;
};

template <bool FULL>
struct __align__(16) Smem {
    float B[2][ROWS][CST];             // B~ rows (u, r), by chunk parity
    float C[FULL ? ROWS : 1][CST];     // C~ rows (t, r)
    float XT[P][SST];                  // x_u mimo_x[p, r], [p][(u, r)]
    float S[FULL ? ROWS : 1][SST];     // masked scores, rows (t, r), columns (u, r')
    float part[GR][NH];                // sum of dt theta per token group, per pair
    Tok tok[3];                        // by chunk mod 3
};

struct Args {
    int B, T, H, G;
    int trap, cplx;
    int64_t rs;
    ProjLayout pl;
    m3_layer_params prm;
    const float* proj;
    const float* dt_scale;
    const float* Bn;  // [B*T][G][NR]
    const float* Cn;
    float* y_out;     // [B][T][H*P]
    float* h_final;   // [B][H][P][N] or null
    float* angle;     // [B][H][NH] or null
    float* prev_bx;   // [B][H][P][N] or null
    // With stage set, the per-token operands the layer backward reads (the staged fp32
    // layer's layouts, token row (b T + t) H + h): dt, A, angles, x_r, x_g, x_b, B~, B~ of
    // the previous token, C~ and y before the gate.
    Fp32LayerParts st;
    int stage;
    // With hs_every > 0 the walk also stores its chunk-start states into st.Hs in the layer
    // backward's chunking: the state entering every hs_every-th chunk k at entry k / hs_every
    // of (B, hs_K + 1, H, P, N) (the zero start at entry 0), and the final state at entry hs_K.
    int hs_every, hs_K;
    // segments of the sequence (segs = 1: none), of which a launch takes lo .. hi - 1, and the
    // state pass's results, per segment but the last and (batch, head): end state
    // [slot][wave][tile][lane] (seg_combine_f32 turns it into the state entering the next
    // segment; that entering segment e is in slot (e - 1) % slots), log-decay, RoPE angle increments
    int segs;
    int lo, hi, slots;
    f32x4* hseg;
    float* lseg;
    float* aseg;
};

constexpr int kSeg0 = 128;  // tokens of the first segments (seg_start)

__device__ __forceinline__ f32x4 mfma4(float a, float b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// exp through the hardware exp2 (relative error ~1e-7 for the arguments here: decays and
// gate inputs), and SiLU on it
__device__ __forceinline__ float exp_hw(float x) { return __builtin_amdgcn_exp2f(x * kLog2e); }
__device__ __forceinline__ float silu_hw(float x) { return x * __builtin_amdgcn_rcpf(1.f + exp_hw(-x)); }

__global__ __launch_bounds__(256) void bc_norm_f32(const float* __restrict__ proj, int64_t rs,
                                                   int64_t offB, int64_t offC, int G,
                                                   int64_t nrows, float eps,
                                                   const float* __restrict__ wB,
                                                   const float* __restrict__ biasB,
                                                   const float* __restrict__ wC,
                                                   const float* __restrict__ biasC,
                                                   float* __restrict__ Bn, float* __restrict__ Cn) {
    const int lane = threadIdx.x & 63;
    const int64_t tg = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (tg >= nrows) return;
    const int64_t tok = tg / G;
    const int g = (int)(tg % G);
    const float* row = proj + tok * rs;
    const int e = 4 * lane;
    const f32x4 vb = *reinterpret_cast<const f32x4*>(row + offB + (int64_t)g * NR + e);
    const f32x4 vc = *reinterpret_cast<const f32x4*>(row + offC + (int64_t)g * NR + e);
    const f32x4 wb = *reinterpret_cast<const f32x4*>(wB + e);
    const f32x4 wc = *reinterpret_cast<const f32x4*>(wC + e);
    const f32x4 bb = *reinterpret_cast<const f32x4*>(biasB + (int64_t)g * NR + e);
    const f32x4 bc = *reinterpret_cast<const f32x4*>(biasC + (int64_t)g * NR + e);
    float sb = 0.f, sc = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        sb += vb[j] * vb[j];
        sc += vc[j] * vc[j];
    }
    sb = lane_sum<64>(sb);
    sc = lane_sum<64>(sc);
    const float rb = rsqrtf(sb / NR + eps), rc = rsqrtf(sc / NR + eps);
    f32x4 ob, oc;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        ob[j] = vb[j] * rb * wb[j] + bb[j];
        oc[j] = vc[j] * rc * wc[j] + bc[j];
    }
    *reinterpret_cast<f32x4*>(Bn + tg * NR + e) = ob;
    *reinterpret_cast<f32x4*>(Cn + tg * NR + e) = oc;
}

__device__ __forceinline__ float ld_b32(const __amdgpu_buffer_rsrc_t& r, int off, int so) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, so, 0));
}
__device__ __forceinline__ f32x4 ld_b128(const __amdgpu_buffer_rsrc_t& r, int off, int so) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, so, 0));
}

// sin and cos of |x| <= kSincosMax: x minus the nearest multiple of pi/2, in three steps of a
// split pi/2 (Cody and Waite), then the Cephes library's minimax polynomials on [-pi/4, pi/4].
// Straight-line, so that a thread's angles interleave; sincosf spends about four times the
// cycles on its range branches. Largest error over the range 7.1e-8, rms 1.7e-8 (float rounding
// of the exact value: 6e-8, 1.5e-8).
constexpr float kSincosMax = 1e5f;
__device__ __forceinline__ void sincos_small(float x, float& s, float& c) {
    const float k = rintf(x * 0.636619772f);
    float r = fmaf(-k, 1.57079637e+00f, x);
    r = fmaf(-k, -4.37113883e-08f, r);
    r = fmaf(-k, -1.71512451e-15f, r);
    const float r2 = r * r;
    float p = fmaf(r2, -1.9515295891e-4f, 8.3321608736e-3f);
    p = fmaf(p, r2, -1.6666654611e-1f);
    const float sr = fmaf(p * r2, r, r);
    float q = fmaf(r2, 2.443315711809948e-5f, -1.388731625493765e-3f);
    q = fmaf(q, r2, 4.166664568298827e-2f);
    q = fmaf(q, r2, -0.5f);
    const float cr = fmaf(q, r2, 1.f);
    const int n = (int)k;
    const unsigned ss = n & 1 ? __builtin_bit_cast(unsigned, cr) : __builtin_bit_cast(unsigned, sr);
    const unsigned cc = n & 1 ? __builtin_bit_cast(unsigned, sr) : __builtin_bit_cast(unsigned, cr);
    s = __builtin_bit_cast(float, ss ^ ((unsigned)(n & 2) << 30));
    c = __builtin_bit_cast(float, cc ^ ((unsigned)((n + 1) & 2) << 30));
}

template <bool FULL>
__global__ __launch_bounds__(THREADS, 3) void ssd_f32(Args a) {
    __shared__ Smem<FULL> sm;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int l16 = lane & 15, g16 = lane >> 4;
    const int npairs = a.B * a.H;
    // Segments longest first; within one, consecutive (batch, head) pairs share an XCD.
    const int j0 = blockIdx.x % npairs;
    const int seg = (FULL ? a.hi : min(a.hi, a.segs - 1)) - 1 - (int)(blockIdx.x / npairs);
    const int bh = (npairs % 8 == 0) ? (j0 % 8) * (npairs / 8) + j0 / 8 : j0;
    const int b = bh / a.H, h = bh % a.H;
    const int grp = h / (a.H / a.G);
    const int T = a.T;
    const int tbeg = (int)seg_start(seg, kSeg0);
    const int tend = seg + 1 < a.segs ? (int)seg_start(seg + 1, kSeg0) : T;
    const int K = (tend - tbeg + Q - 1) / Q;
    const int k0 = tbeg / Q;              // the segment's first chunk in the sequence
    const int KT = (T + Q - 1) / Q;
    const float Ah = -expf(a.prm.A_log[h]);
    const float* proj = a.proj + (int64_t)b * T * a.rs;
    const int rb = (int)a.rs * 4;         // bytes of a proj row
    // Reads of a chunk go through buffer resources that start at its first token and end at the
    // sequence's last: tokens past the end read as zero.
    auto chunk_rsrc = [&](const void* base, int kk, int64_t row_bytes) {
        const int64_t s0 = tbeg + (int64_t)kk * Q;
        return make_rsrc(reinterpret_cast<const char*>(base) + (s0 < T ? s0 * row_bytes : 0),
                         s0 < T ? (T - s0) * row_bytes : 0);
    };

    if (wave < CW) {
        // =============================== column waves ===============================
        const int p = 16 * wave + l16;
        f32x4 hacc[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) hacc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (FULL && seg > 0) {
            const f32x4* hs = a.hseg + (((int64_t)((seg - 1) % a.slots) * npairs + bh) * CW + wave) * (NT * 64) + lane;
#pragma unroll
            for (int t = 0; t < NT; ++t) hacc[t] = hs[t * 64];
        }
        float mz[R], md[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            mz[r] = a.prm.mimo_z[(h * P + p) * R + r];
            md[r] = a.prm.mimo_down[(h * P + p) * R + r];
        }
        // chunk-start states for the layer backward: entry e of (B, hs_K + 1, H, P, N), this
        // lane's column
        auto hs_entry = [&](int e) {
            return a.st.Hs + (((int64_t)b * (a.hs_K + 1) + e) * a.H + h) * (P * N) + (int64_t)p * N + 4 * g16;
        };
        if (FULL && a.hs_every > 0 && seg == 0) {  // the zero start state
            float* hk = hs_entry(0);
#pragma unroll
            for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4*>(hk + 16 * t) = hacc[t];
        }
        float ldec = 0.f;  // log of the segment's decay (state pass)
        __syncthreads();  // token scalars of chunks 0 and 1
        __syncthreads();  // angle sums of chunk 0
        __syncthreads();  // tiles of chunk 0

        for (int k = 0; k < K; ++k) {
            const int s0 = tbeg + k * Q;
            const Tok& tk = sm.tok[k % 3];
            const float (&sB)[ROWS][CST] = sm.B[k & 1];
            // ---- scores ----
            float zv[FULL ? 4 : 1][2];
            f32x4 y[FULL ? 4 : 1], gz[FULL ? 4 : 1];
            if constexpr (FULL) {
                const __amdgpu_buffer_rsrc_t rp = chunk_rsrc(proj, k, rb);
                const int zoff = 2 * g16 * rb + ((int)a.pl.z + h * P + p) * 4;
#pragma unroll
                for (int tt = 0; tt < 4; ++tt) {
                    zv[tt][0] = ld_b32(rp, zoff, 8 * tt * rb);
                    zv[tt][1] = ld_b32(rp, zoff, (8 * tt + 1) * rb);
                    y[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
                f32x4 A[2][4];
                auto load_c = [&](int t) {
#pragma unroll
                    for (int tt = 0; tt < 4; ++tt) A[t & 1][tt] = *reinterpret_cast<const f32x4*>(&sm.C[16 * tt + l16][16 * t + 4 * g16]);
                };
                load_c(0);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    if (t + 1 < NT) load_c(t + 1);
                    M3_FENCE();
#pragma unroll
                    for (int v = 0; v < 4; ++v)
#pragma unroll
                        for (int tt = 0; tt < 4; ++tt) y[tt] = mfma4(A[t & 1][tt][v], hacc[t][v], y[tt]);
                }
                // gate factors of the two ranks
#pragma unroll
                for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const float z = zv[tt][q];
                        gz[tt][2 * q] = md[0] * silu_hw(z * mz[0]);
                        gz[tt][2 * q + 1] = md[1] * silu_hw(z * mz[1]);
                    }
#pragma unroll
                for (int tt = 0; tt < 4; ++tt) {
                    const f32x2 e = *reinterpret_cast<const f32x2*>(&tk.ec[8 * tt + 2 * g16]);
                    y[tt][0] *= e[0];
                    y[tt][1] *= e[0];
                    y[tt][2] *= e[1];
                    y[tt][3] *= e[1];
                }
            }
            M3_FENCE();
            __syncthreads();
            // ---- update ----
            f32x4 X[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) X[s] = *reinterpret_cast<const f32x4*>(&sm.XT[p][16 * s + 4 * g16]);
            if constexpr (FULL) {
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    f32x4 A[4];
#pragma unroll
                    for (int tt = s; tt < 4; ++tt) A[tt] = *reinterpret_cast<const f32x4*>(&sm.S[16 * tt + l16][16 * s + 4 * g16]);
#pragma unroll
                    for (int v = 0; v < 4; ++v)
#pragma unroll
                        for (int tt = s; tt < 4; ++tt) y[tt] = mfma4(A[tt][v], X[s][v], y[tt]);
                }
                // gate and MIMO-down: rows 4 g16 + 2 q + r of row block tt are (t, r); stores past
                // the sequence's end fall outside the resource
                const __amdgpu_buffer_rsrc_t ro = chunk_rsrc(a.y_out + (int64_t)b * T * a.H * P, k, (int64_t)a.H * P * 4);
                const int ob = a.H * P * 4, ooff = 2 * g16 * ob + (h * P + p) * 4;
#pragma unroll
                for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const float o = gz[tt][2 * q] * y[tt][2 * q] + gz[tt][2 * q + 1] * y[tt][2 * q + 1];
                        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, o), ro, ooff, (8 * tt + q) * ob, 0);
                    }
            }
            {
                const float dec = tk.ec[Q - 1];
                if constexpr (!FULL) ldec += tk.cend;
#pragma unroll
                for (int t = 0; t < NT; ++t) hacc[t] *= dec;
                // rows 4 g16 + v of k-step i = 4 s + v
                float A[2][NT], xw[4][4];
                auto load_b = [&](int i) {
#pragma unroll
                    for (int t = 0; t < NT; ++t) A[i & 1][t] = sB[16 * (i / 4) + 4 * g16 + i % 4][16 * t + l16];
                };
                load_b(0);
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const f32x2 w = *reinterpret_cast<const f32x2*>(&tk.w[8 * s + 2 * g16]);
#pragma unroll
                    for (int v = 0; v < 4; ++v) xw[s][v] = X[s][v] * w[v / 2];
                }
#pragma unroll
                for (int i = 0; i < ROWS / 4; ++i) {
                    if (i + 1 < ROWS / 4) load_b(i + 1);
                    M3_FENCE();
#pragma unroll
                    for (int t = 0; t < NT; ++t) hacc[t] = mfma4(A[i & 1][t], xw[i / 4][i % 4], hacc[t]);
                }
            }
            if constexpr (FULL) {
                if (a.stage) {
#pragma unroll
                    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
                        for (int q = 0; q < 2; ++q) {
                            const int st = s0 + 8 * tt + 2 * g16 + q;
                            if (st < T)
                                *reinterpret_cast<f32x2*>(a.st.ys + ((((int64_t)b * T + st) * a.H + h) * P + p) * R) =
                                    f32x2{y[tt][2 * q], y[tt][2 * q + 1]};
                        }
                }
            }
            // The state entering the next chunk for the layer backward. The walk folds the beta
            // term of the next chunk's first token into this chunk (b_{Q-1} B~_{Q-1} x_{Q-1}^T); the
            // chunk kernels count it in the next chunk, so it is taken out of the stored state
            // (b = 0 without the trapezoid).
            if (FULL && a.hs_every > 0 && (k0 + k + 1) % a.hs_every == 0 && k0 + k + 1 < KT) {
                const float bq = tk.bv[Q - 1];
                const float x0 = bq * sm.XT[p][2 * (Q - 1)], x1 = bq * sm.XT[p][2 * (Q - 1) + 1];
                float* hk = hs_entry((k0 + k + 1) / a.hs_every);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const f32x4 b0 = *reinterpret_cast<const f32x4*>(&sB[2 * (Q - 1)][16 * t + 4 * g16]);
                    const f32x4 b1 = *reinterpret_cast<const f32x4*>(&sB[2 * (Q - 1) + 1][16 * t + 4 * g16]);
                    *reinterpret_cast<f32x4*>(hk + 16 * t) = hacc[t] - (b0 * x0 + b1 * x1);
                }
            }
            __syncthreads();
        }
        if constexpr (FULL) {
            if (tend == T) {
                if (a.hs_every > 0) {
                    float* hk = hs_entry(a.hs_K);
#pragma unroll
                    for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4*>(hk + 16 * t) = hacc[t];
                }
                if (a.h_final) {
                    float* hf = a.h_final + (int64_t)bh * P * N + (int64_t)p * N + 4 * g16;
#pragma unroll
                    for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4*>(hf + 16 * t) = hacc[t];
                }
            }
        } else {
            f32x4* hs = a.hseg + (((int64_t)(seg % a.slots) * npairs + bh) * CW + wave) * (NT * 64) + lane;
#pragma unroll
            for (int t = 0; t < NT; ++t) hs[t * 64] = hacc[t];
            if (wave == 0 && lane == 0) a.lseg[(int64_t)seg * npairs + bh] = ldec;
        }
    } else {
        // =============================== helper waves ===============================
        const int hw = wave - CW, htid = tid - 64 * CW;
        const float Dh = a.prm.D[h];
        const float dtb = a.prm.dt_bias[h];
        const int64_t nrs = (int64_t)a.G * NR;  // B^ / C^ token stride
        const int nb = (int)nrs * 4;
        const float* Bn = a.Bn + (int64_t)b * T * nrs + (int64_t)grp * NR;
        const float* Cn = a.Cn + (int64_t)b * T * nrs + (int64_t)grp * NR;
        const bool stage = FULL && a.stage;
        if (stage && htid == 0) a.st.A[h] = Ah;
        // rotation jobs: RoPE pairs 2 hl, 2 hl + 1 (columns 4 hl ..) of tokens tg TPT + m; a pair's
        // words are (n=2i, r0) (2i, r1) (2i+1, r0) (2i+1, r1)
        const int hl = lane % LPT, tg = htid / LPT;
        f32x4 pb[TPT][2], pc[FULL ? TPT : 1][2];
        auto load_bc = [&](int kk) {
            const int off = tg * TPT * nb + 32 * hl;
            const __amdgpu_buffer_rsrc_t r = chunk_rsrc(Bn, kk, nb);
#pragma unroll
            for (int m = 0; m < TPT; ++m) {
                pb[m][0] = ld_b128(r, off, m * nb);
                pb[m][1] = ld_b128(r, off + 16, m * nb);
            }
            if constexpr (FULL) {
                const __amdgpu_buffer_rsrc_t rc = chunk_rsrc(Cn, kk, nb);
#pragma unroll
                for (int m = 0; m < TPT; ++m) {
                    pc[m][0] = ld_b128(rc, off, m * nb);
                    pc[m][1] = ld_b128(rc, off + 16, m * nb);
                }
            }
        };
        // X jobs: column xp, tokens xt0 .. xt0 + XTOK - 1
        const int xp = htid % P, xt0 = (htid / P) * XTOK;
        const float mx0 = a.prm.mimo_x[(h * P + xp) * R], mx1 = a.prm.mimo_x[(h * P + xp) * R + 1];
        float pxv[XTOK];
        auto load_xv = [&](int kk) {
            const __amdgpu_buffer_rsrc_t r = chunk_rsrc(proj, kk, rb);
            const int off = xt0 * rb + ((int)a.pl.x + h * P + xp) * 4;
#pragma unroll
            for (int m = 0; m < XTOK; ++m) pxv[m] = ld_b32(r, off, m * rb);
        };
        f32x2 pth[TPT] = {};  // theta of the rotation jobs' pairs
        auto load_theta = [&](int kk) {
            if (!a.cplx) return;  // no theta columns
            const __amdgpu_buffer_rsrc_t r = chunk_rsrc(proj, kk, rb);
            const int off = tg * TPT * rb + ((int)a.pl.theta + 2 * hl) * 4;
#pragma unroll
            for (int m = 0; m < TPT; ++m) pth[m] = f32x2{ld_b32(r, off, m * rb), ld_b32(r, off + 4, m * rb)};
        };
        // token scalars: lane t = token t of the chunk (the last helper)
        float rdt0 = 0.f, rdt1 = 0.f, rlam0 = 0.f, rlam1 = 0.f, sc0 = 1.f, sc1 = 1.f;
        auto load_tokens = [&](int kk) {
            const __amdgpu_buffer_rsrc_t r = chunk_rsrc(proj, kk, rb);
            const int off = lane * rb + h * 4;
            rdt0 = ld_b32(r, off, (int)a.pl.dt * 4);
            rdt1 = ld_b32(r, off + rb, (int)a.pl.dt * 4);
            if (a.trap) {
                rlam0 = ld_b32(r, off, (int)a.pl.lam * 4);
                rlam1 = ld_b32(r, off + rb, (int)a.pl.lam * 4);
            }
            if (a.dt_scale) {
                const __amdgpu_buffer_rsrc_t rd = chunk_rsrc(a.dt_scale + (int64_t)b * T * a.H, kk, (int64_t)a.H * 4);
                sc0 = ld_b32(rd, (lane * a.H + h) * 4, 0);
                sc1 = ld_b32(rd, ((lane + 1) * a.H + h) * 4, 0);
            }
        };
        auto prep_tokens = [&](int kk) {
            const int s0 = tbeg + kk * Q, t = lane;
            const bool v0 = t < Q && s0 + t < T, v1 = t < Q && s0 + t + 1 < T;
            const float dt0 = v0 ? softplus_f(rdt0 + dtb) * sc0 : 0.f;
            const float dt1 = v1 ? softplus_f(rdt1 + dtb) * sc1 : 0.f;
            const float lam0 = v0 && a.trap ? sigmoid_f(rlam0) : 1.f;
            const float lam1 = v1 && a.trap ? sigmoid_f(rlam1) : 1.f;
            const float c = wave_incl_scan(Ah * dt0);
            const float cend = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, c), Q - 1));
            Tok& tk = sm.tok[kk % 3];
            if (t < Q) {
                const float av = a.trap ? lam0 * dt0 : dt0;
                const float bv = a.trap ? (1.f - lam1) * dt1 : 0.f;
                tk.c[t] = c;
                tk.ec[t] = exp_hw(c);
                tk.av[t] = av;
                tk.bv[t] = bv;
                tk.w[t] = exp_hw(cend - c) * (av + bv);
                tk.dt[t] = dt0;
                tk.lam[t] = lam0;
                tk.sb[t] = a.trap ? (1.f - lam1) * expf(Ah * dt1) : 0.f;
                if (stage && v0 && s0 + t < tend) a.st.dt[((int64_t)b * T + s0 + t) * a.H + h] = dt0;
            }
            if (t == 0) tk.cend = cend;
        };
        // this thread's sums of dt theta over its token group, chunk kk
        auto angle_sums = [&](int kk) {
            if (!a.cplx) return;
            const Tok& tk = sm.tok[kk % 3];
            f32x2 ps = f32x2{0.f, 0.f};
#pragma unroll
            for (int m = 0; m < TPT; ++m) ps += pth[m] * tk.dt[tg * TPT + m];
            *reinterpret_cast<f32x2*>(&sm.part[tg][2 * hl]) = ps;
        };
        f32x2 phi_run = f32x2{0.f, 0.f};  // pair angles at the start of the chunk to rotate next
        if (FULL && a.cplx)
#pragma unroll 4
            for (int j = 0; j < seg; ++j)
                phi_run += *reinterpret_cast<const f32x2*>(a.aseg + ((int64_t)j * npairs + bh) * NH + 2 * hl);
        // sin / cos of chunk kk's pairs: phi_t[i] = phi_{t-1}[i] - dt_t theta_t[i]
        // (mamba3/mamba3.py:160-162)
        f32x2 cs[TPT], sn[TPT];
        auto angles = [&](int kk) {
            const Tok& tk = sm.tok[kk % 3];
            f32x2 ph = phi_run;
            if (a.cplx) {
                f32x2 pp[GR], run = phi_run;
#pragma unroll
                for (int g = 0; g < GR; ++g) pp[g] = *reinterpret_cast<const f32x2*>(&sm.part[g][2 * hl]);
                M3_FENCE();
#pragma unroll
                for (int g = 0; g < GR; ++g) {
                    if (g == tg) ph = run;
                    run -= pp[g];
                }
                phi_run = run;
            }
            f32x2 pm[TPT];
            bool small = true;
#pragma unroll
            for (int m = 0; m < TPT; ++m) {
                const int t = tg * TPT + m, st = tbeg + kk * Q + t;
                if (a.cplx) ph -= pth[m] * tk.dt[t];
                pm[m] = ph;
                small &= fabsf(ph[0]) <= kSincosMax && fabsf(ph[1]) <= kSincosMax;
                if (stage && st < T)
                    *reinterpret_cast<f32x2*>(a.st.phi + (((int64_t)b * T + st) * a.H + h) * NH + 2 * hl) = ph;
            }
            // (without complex parameters the angles are 0: cos 1, sin 0)
            if (small) {
#pragma unroll
                for (int m = 0; m < TPT; ++m)
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        float s, c;
                        sincos_small(pm[m][e], s, c);
                        sn[m][e] = s;
                        cs[m][e] = c;
                    }
            } else {
#pragma unroll 1
                for (int m = 0; m < TPT; ++m)
#pragma unroll 1
                    for (int e = 0; e < 2; ++e) {
                        float s, c;
                        sincosf(pm[m][e], &s, &c);
                        sn[m][e] = s;
                        cs[m][e] = c;
                    }
            }
        };
        // X^T columns (t, r) = x_t * mimo_x[p, r] (mamba3/mamba3.py:210) of chunk kk
        auto write_x = [&](int kk) {
            const Tok& tk = sm.tok[kk % 3];
            f32x4 xo[XTOK / 2];
#pragma unroll
            for (int m = 0; m < XTOK; ++m) {
                const int t = xt0 + m, st = tbeg + kk * Q + t;
                const f32x2 xr = f32x2{pxv[m] * mx0, pxv[m] * mx1};
                xo[m / 2][2 * (m % 2)] = xr[0];
                xo[m / 2][2 * (m % 2) + 1] = xr[1];
                if (stage && st < T) {
                    // x_r, x_g = lambda_t x_r and x_b of the next token (mamba3/mamba3.py:210-224)
                    const int64_t e = ((((int64_t)b * T + st) * a.H + h) * P + xp) * R;
                    *reinterpret_cast<f32x2*>(a.st.xr + e) = xr;
                    *reinterpret_cast<f32x2*>(a.st.xg + e) = xr * tk.lam[t];
                    if (a.trap) {
                        if (st + 1 < T) *reinterpret_cast<f32x2*>(a.st.xb + e + (int64_t)a.H * P * R) = xr * tk.sb[t];
                        if (st == 0) *reinterpret_cast<f32x2*>(a.st.xb + e) = f32x2{0.f, 0.f};
                    }
                }
            }
#pragma unroll
            for (int v = 0; v < XTOK / 2; ++v) *reinterpret_cast<f32x4*>(&sm.XT[xp][xt0 * R + 4 * v]) = xo[v];
        };
        // rotated C~ / B~ rows of the words in hand (words of tokens past the end are zero),
        // chunk kk
        auto write_tiles = [&](int kk) {
            float (&sB)[ROWS][CST] = sm.B[kk & 1];
#pragma unroll
            for (int m = 0; m < TPT; ++m) {
                const int t = tg * TPT + m, st = tbeg + kk * Q + t;
                const f32x2 c = cs[m], s = sn[m];
                // rank r: words r (n even) and 2 + r (n odd) of each pair
                auto turn = [&](const f32x4 (&v)[2], int r) {
                    return f32x4{v[0][r] * c[0] - v[0][2 + r] * s[0], v[0][r] * s[0] + v[0][2 + r] * c[0],
                                 v[1][r] * c[1] - v[1][2 + r] * s[1], v[1][r] * s[1] + v[1][2 + r] * c[1]};
                };
                const f32x4 b0 = turn(pb[m], 0), b1 = turn(pb[m], 1);
                *reinterpret_cast<f32x4*>(&sB[2 * t][4 * hl]) = b0;
                *reinterpret_cast<f32x4*>(&sB[2 * t + 1][4 * hl]) = b1;
                if constexpr (FULL) {
                    const f32x4 c0 = turn(pc[m], 0), c1 = turn(pc[m], 1);
                    *reinterpret_cast<f32x4*>(&sm.C[2 * t][4 * hl]) = c0;
                    *reinterpret_cast<f32x4*>(&sm.C[2 * t + 1][4 * hl]) = c1;
                    if (stage && st < T) {
                        const int64_t tk = ((int64_t)b * T + st) * a.H + h;
                        const f32x4 bl = f32x4{b0[0], b1[0], b0[1], b1[1]}, bu = f32x4{b0[2], b1[2], b0[3], b1[3]};
                        f32x4* q = reinterpret_cast<f32x4*>(a.st.Bt + tk * NR + 8 * hl);
                        q[0] = bl;
                        q[1] = bu;
                        q = reinterpret_cast<f32x4*>(a.st.Ct + tk * NR + 8 * hl);
                        q[0] = f32x4{c0[0], c1[0], c0[1], c1[1]};
                        q[1] = f32x4{c0[2], c1[2], c0[3], c1[3]};
                        if (a.trap) {  // B_b[t + 1] = B~[t]
                            if (st + 1 < T) {
                                q = reinterpret_cast<f32x4*>(a.st.Bb + (tk + a.H) * NR + 8 * hl);
                                q[0] = bl;
                                q[1] = bu;
                            }
                            if (st == 0) {
                                q = reinterpret_cast<f32x4*>(a.st.Bb + tk * NR + 8 * hl);
                                q[0] = q[1] = f32x4{0.f, 0.f, 0.f, 0.f};
                            }
                        }
                    }
                }
            }
        };
        const bool token_wave = hw == HW - 1;

        // Prologue: chunks 0 and 1's token scalars, chunk 0's tiles, chunk 1's reads (chunks past
        // the end read as zero).
        load_bc(0);
        load_xv(0);
        load_theta(0);
        if (hw >= HW - 2) {
            load_tokens(hw - (HW - 2));
            prep_tokens(hw - (HW - 2));
            if (token_wave) load_tokens(2);
        }
        __syncthreads();
        angle_sums(0);
        __syncthreads();
        angles(0);
        write_tiles(0);
        load_bc(1);
        load_theta(1);
        __syncthreads();

        for (int k = 0; k < K; ++k) {
            const bool more = k + 1 < K;
            // ---- scores ----
            if constexpr (FULL) {
                // causal score tiles (ti, ui), ui <= ti: helpers 0-3 take (3, 0..3), 4-6 (2, 0..2) and
                // (1, 0), (1, 1), (0, 0); lane: u-rows 16 ui + 4 g16 + v, t-row 16 ti + l16
                const Tok& tk = sm.tok[k % 3];
                const float (&sB)[ROWS][CST] = sm.B[k & 1];
                const int nt = hw < 4 ? 1 : token_wave ? 0 : 2;
#pragma unroll 1
                for (int c = 0; c < nt; ++c) {
                    const int ti = hw < 4 ? 3 : c == 0 ? 2 : hw == 6 ? 0 : 1;
                    const int ui = hw == 6 && c == 1 ? 0 : hw & 3;
                    f32x4 s0 = f32x4{0.f, 0.f, 0.f, 0.f}, s1 = s0;  // even and odd k-steps
                    f32x4 A[2][2], B[2][2];
                    auto load_s = [&](int s) {
#pragma unroll
                        for (int j = 0; j < 2; ++j) {
                            A[s & 1][j] = *reinterpret_cast<const f32x4*>(&sB[16 * ui + l16][32 * s + 16 * j + 4 * g16]);
                            B[s & 1][j] = *reinterpret_cast<const f32x4*>(&sm.C[16 * ti + l16][32 * s + 16 * j + 4 * g16]);
                        }
                    };
                    load_s(0);
#pragma unroll
                    for (int s = 0; s < N / 32; ++s) {
                        if (s + 1 < N / 32) load_s(s + 1);
                        M3_FENCE();
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            s0 = mfma4(A[s & 1][0][v], B[s & 1][0][v], s0);
                            s1 = mfma4(A[s & 1][1][v], B[s & 1][1][v], s1);
                        }
                    }
                    s0 += s1;
                    // the lane's rows are two tokens u, u + 1; masked pairs get weight 0 (their
                    // exponent is capped, so no overflow meets the 0)
                    const int trow = 16 * ti + l16, t = trow >> 1, u = 8 * ui + 2 * g16;
                    const float ct = tk.c[t];
                    const f32x2 cu = *reinterpret_cast<const f32x2*>(&tk.c[u]);
                    const f32x2 au = *reinterpret_cast<const f32x2*>(&tk.av[u]);
                    const f32x2 bu = *reinterpret_cast<const f32x2*>(&tk.bv[u]);
                    float f[2];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const float wu = u + e < t ? au[e] + bu[e] : u + e == t ? au[e] : 0.f;
                        f[e] = exp_hw(fminf(ct - cu[e], 0.f)) * wu;
                    }
                    f32x4 sv;
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        sv[v] = u + v / 2 <= t ? s0[v] * f[v / 2] : 0.f;
                        if (2 * u + v == trow) sv[v] += Dh;
                    }
                    *reinterpret_cast<f32x4*>(&sm.S[trow][16 * ui + 4 * g16]) = sv;
                }
            }
            write_x(k);
            load_xv(k + 1);
            if (more) angle_sums(k + 1);
            if (token_wave) {
                prep_tokens(k + 2);
                load_tokens(k + 3);
            }
            __syncthreads();
            // ---- update ----
            if (more) {
                angles(k + 1);
                write_tiles(k + 1);
                load_bc(k + 2);
                load_theta(k + 2);
            }
            __syncthreads();
        }
        // phi_run is the angle after the last chunk
        if constexpr (FULL) {
            if (a.angle && tend == T && htid < LPT) {
                float* ang = a.angle + (int64_t)bh * NH + 2 * hl;
                ang[0] = phi_run[0];
                ang[1] = phi_run[1];
            }
            if (a.prev_bx && tend == T) {
                // B~_{T-1} x_r,{T-1}^T from the last chunk's tiles
                const int ul = T - 1 - tbeg - (K - 1) * Q;
                for (int i = htid; i < P * N / 4; i += HT) {
                    const int pp = i / (N / 4), n = 4 * (i % (N / 4));
                    const f32x4 b0 = *reinterpret_cast<const f32x4*>(&sm.B[(K - 1) & 1][2 * ul][n]);
                    const f32x4 b1 = *reinterpret_cast<const f32x4*>(&sm.B[(K - 1) & 1][2 * ul + 1][n]);
                    *reinterpret_cast<f32x4*>(a.prev_bx + ((int64_t)bh * P + pp) * N + n) =
                        b0 * sm.XT[pp][2 * ul] + b1 * sm.XT[pp][2 * ul + 1];
                }
            }
        } else {
            if (htid < LPT)
                *reinterpret_cast<f32x2*>(a.aseg + ((int64_t)seg * npairs + bh) * NH + 2 * hl) = phi_run;
        }
    }
}

// Turns the segments' end states (from a zero start, each in its own RoPE frame) into the
// states entering the next segments, in place: one thread per four state rows of a column.
__global__ __launch_bounds__(256) void seg_combine_f32(Args a) {
    constexpr int PER = CW * NT * 64;  // entries per (batch, head)
    const int npairs = a.B * a.H;
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= (int64_t)npairs * PER) return;
    const int bh = (int)(e / PER), t = (int)(e % (NT * 64)) / 64, g16 = (int)(e % 64) / 16;
    const int i = (16 * t + 4 * g16) / 2;  // first RoPE pair
    f32x4 h = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x2 phi = f32x2{0.f, 0.f};
    auto slot = [&](int j) { return a.hseg + (int64_t)(j % a.slots) * npairs * PER + e; };
    auto angle_inc = [&](int j) {
        return *reinterpret_cast<const f32x2*>(a.aseg + ((int64_t)j * npairs + bh) * NH + i);
    };
    if (a.lo > 0) h = *slot(a.lo - 1);
    for (int j = 0; j < a.lo; ++j) phi += angle_inc(j);
    const int hi = min(a.hi, a.segs - 1);
#pragma unroll 2
    for (int j = a.lo; j < hi; ++j) {
        f32x4* hj = slot(j);
        const f32x4 v = *hj;
        const f32x2 inc = angle_inc(j);
        const float dec = expf(a.lseg[(int64_t)j * npairs + bh]);
        float s0, c0, s1, c1;
        sincosf(phi[0], &s0, &c0);
        sincosf(phi[1], &s1, &c1);
        // (the first segment's state is in the sequence's frame already)
        h = j == 0 ? v : h * dec + f32x4{v[0] * c0 - v[1] * s0, v[0] * s0 + v[1] * c0,
                                         v[2] * c1 - v[3] * s1, v[2] * s1 + v[3] * c1};
        *hj = h;
        phi += inc;
    }
}

// Segments of a sequence, by its heads and tokens alone: not by the batch, so that a sequence
// gives the same bits alone and in any batch. The state pass costs about half a walk, so segments
// pay while the (batch, head) pairs leave more than half of the 256 CUs idle, and more pairs pay
// for it. us per call at 24 heads, cut / uncut: (1, 300) 70 / 94, (1, 1000) 125 / 276, (4, 600)
// 136 / 169, (4, 4096) 681 / 1085; but (8, 300) 157 / 97, (8, 1000) 354 / 279, (8, 2048) 670 / 563.
// At the line, one sequence of 126 heads, 600 and 2,048 tokens: 177 / 169, 444 / 535.
int segments(const m3_layer_desc& d) { return d.nheads < 128 ? seg_count(d.seqlen, kSeg0) : 1; }

SegSizes seg_sizes(const m3_layer_desc& d, bool rows) {
    return {rows ? (size_t)d.seqlen * d.ngroups * NR * sizeof(float) : 0, (size_t)d.nheads * P * N * sizeof(float),
            d.nheads * sizeof(float), (size_t)d.nheads * NH * sizeof(float)};
}

}  // namespace f32k

static bool fused_fp32_shape_ok(const m3_layer_desc& d, const void* proj, const void* y_out,
                                const void* h_final, const void* prev_bx) {
    if (d.dtype != M3_DTYPE_F32) return false;
    if (d.d_state != f32k::N || d.headdim != f32k::P || d.mimo_rank != f32k::R) return false;
    const ProjLayout pl = proj_layout(d);
    // a chunk's rows are addressed with 32-bit byte offsets
    if (d.proj_row_stride >= (1 << 22) || (int64_t)d.ngroups * f32k::NR >= (1 << 22) || d.nheads >= (1 << 18))
        return false;
    // 16-byte reads of the B / C rows
    if (d.proj_row_stride % 4 != 0 || pl.x % 4 != 0 || pl.z % 4 != 0 || pl.B % 4 != 0 || pl.C % 4 != 0)
        return false;
    auto al16 = [](const void* ptr) { return reinterpret_cast<uintptr_t>(ptr) % 16 == 0; };
    if (!al16(proj) || !al16(y_out) || !al16(h_final) || !al16(prev_bx)) return false;
    return true;
}

bool fused_fp32_prefill_supported(const m3_layer_desc& d, const void* proj, const void* y_out,
                                  const void* h_final, const void* prev_bx) {
    return !(d.flags & M3_FLAG_FOR_BACKWARD) && fused_fp32_shape_ok(d, proj, y_out, h_final, prev_bx);
}

bool fused_fp32_train_supported(const m3_layer_desc& d, const void* proj, const void* y_out,
                                const void* h_final, const void* prev_bx) {
    if (!fused_fp32_shape_ok(d, proj, y_out, h_final, prev_bx) || !fp32_layer_supported(d)) return false;
    size_t bytes = 0;
    fp32_layer_scratch(d, nullptr, &bytes);
    return bytes >= fused_fp32_prefill_min_workspace(d);
}

static SegPlan fused_fp32_plan(const m3_layer_desc& d, size_t limit) {
    return plan_segments(d.batch, f32k::segments(d), f32k::seg_sizes(d, true), limit, true);
}
size_t fused_fp32_prefill_workspace(const m3_layer_desc& d) { return fused_fp32_plan(d, SIZE_MAX).total; }
size_t fused_fp32_prefill_min_workspace(const m3_layer_desc& d) { return fused_fp32_plan(d, 0).total; }

// The training forward's parts of the fp32 layer workspace's chunk-kernel region: with room for
// the chunk-start states (Fp32LayerParts::Hs) the C^ rows lie past them and the segments'
// states between the B^ rows and them, else the segments' states follow both rows.
struct TrainRegion {
    size_t cn, seg, room;  // offsets in the region; bytes for the segments' states
    bool hs;
};
static TrainRegion train_region(const m3_layer_desc& d) {
    const size_t rows = al256((size_t)d.batch * d.seqlen * d.ngroups * f32k::NR * sizeof(float));
    size_t bytes = 0;
    fp32_layer_scratch(d, nullptr, &bytes);
    if (!fp32_layer_hs_ok(d)) return {rows, 2 * rows, bytes > 2 * rows ? bytes - 2 * rows : 0, false};
    const size_t off = chunked_fwd_hs_offset(d.batch, d.seqlen, d.nheads, d.headdim, d.d_state, d.mimo_rank,
                                             d.use_trapezoidal != 0);
    return {off + al256(fp32_layer_hs_bytes(d)), rows, off > rows ? off - rows : 0, true};
}

size_t fused_fp32_train_workspace(const m3_layer_desc& d) {
    const SegPlan p = plan_segments(d.batch, f32k::segments(d), f32k::seg_sizes(d, false), SIZE_MAX, false);
    const bool inside = p.segs == 1 || p.total <= train_region(d).room;
    return al256(fp32_layer_workspace(d)) + (inside ? 0 : p.total);
}

// One slice of the batch: B^ rows at bn, C^ rows at cn, the segments' states as the plan lays
// them out from `seg` on.
static int launch_fused_fp32_slice(const m3_layer_desc& d, const m3_layer_params& p, const float* proj,
                                   const float* dt_scale, float* y_out, float* h_final, float* angle,
                                   float* prev_bx, float* bn, float* cn, char* seg, const SegPlan& sp,
                                   hipStream_t stream, const Fp32LayerParts* stage, bool hs) {
    const ProjLayout pl = proj_layout(d);
    const int64_t nrows = (int64_t)d.batch * d.seqlen * d.ngroups;
    int hs_every = 0, hs_K = 0;
    if (hs) {
        const int qb = chunked_chunk_tokens(d.mimo_rank, d.use_trapezoidal != 0);
        if (qb % f32k::Q != 0) return M3_ERR_UNSUPPORTED;
        hs_every = qb / f32k::Q;
        hs_K = (d.seqlen + qb - 1) / qb;
    }
    hipLaunchKernelGGL(f32k::bc_norm_f32, dim3((unsigned)((nrows + 3) / 4)), dim3(256), 0, stream,
                       proj, d.proj_row_stride, pl.B, pl.C, d.ngroups,
                       nrows, d.rms_eps, p.B_norm_w, p.B_bias, p.C_norm_w, p.C_bias, bn, cn);
    f32k::Args a;
    a.B = d.batch; a.T = d.seqlen; a.H = d.nheads; a.G = d.ngroups;
    a.trap = d.use_trapezoidal; a.cplx = d.use_complex;
    a.rs = d.proj_row_stride;
    a.pl = pl;
    a.prm = p;
    a.proj = proj;
    a.dt_scale = dt_scale;
    a.Bn = bn;
    a.Cn = cn;
    a.y_out = y_out;
    a.h_final = h_final;
    a.angle = angle;
    a.prev_bx = prev_bx;
    a.st = stage ? *stage : Fp32LayerParts{};
    a.stage = stage != nullptr;
    a.hs_every = hs_every;
    a.hs_K = hs_K;
    a.segs = sp.segs;
    a.slots = sp.slots;
    a.hseg = reinterpret_cast<f32x4*>(seg + sp.hseg);
    a.lseg = reinterpret_cast<float*>(seg + sp.lseg);
    a.aseg = reinterpret_cast<float*>(seg + sp.aseg);
    const unsigned bh = (unsigned)(d.batch * d.nheads);
    for (a.lo = 0; a.lo < a.segs; a.lo = a.hi) {
        a.hi = std::min(a.segs, a.lo + sp.group);
        const int ns = std::min(a.hi, a.segs - 1) - a.lo;
        if (ns > 0) {
            hipLaunchKernelGGL(f32k::ssd_f32<false>, dim3(bh * ns), dim3(f32k::THREADS), 0, stream, a);
            hipLaunchKernelGGL(f32k::seg_combine_f32,
                               dim3((unsigned)(((int64_t)bh * f32k::P * f32k::N / 4 + 255) / 256)), dim3(256), 0,
                               stream, a);
        }
        hipLaunchKernelGGL(f32k::ssd_f32<true>, dim3(bh * (a.hi - a.lo)), dim3(f32k::THREADS), 0, stream, a);
    }
    return hipGetLastError() == hipSuccess ? M3_OK : M3_ERR_LAUNCH;
}

int launch_fused_fp32_prefill(const m3_layer_desc& d, const m3_layer_params& p, const void* proj,
                              const float* dt_scale, void* y_out, float* h_final, float* angle,
                              float* prev_bx, void* workspace, size_t limit, hipStream_t stream) {
    const SegPlan sp = fused_fp32_plan(d, limit);
    char* ws = reinterpret_cast<char*>(workspace);
    const int64_t T = d.seqlen, H = d.nheads;
    for (int b = 0; b < d.batch; b += sp.batch) {
        m3_layer_desc part = d;
        part.batch = std::min(sp.batch, d.batch - b);
        auto at = [&](auto* q, int64_t per_row) { return q ? q + b * per_row : nullptr; };
        const int st = launch_fused_fp32_slice(
            part, p, reinterpret_cast<const float*>(proj) + b * T * d.proj_row_stride, at(dt_scale, T * H),
            reinterpret_cast<float*>(y_out) + b * T * H * f32k::P, at(h_final, H * f32k::P * f32k::N),
            at(angle, H * f32k::NH), at(prev_bx, H * f32k::P * f32k::N), reinterpret_cast<float*>(ws),
            reinterpret_cast<float*>(ws + sp.rows), ws, sp, stream, nullptr, false);
        if (st != M3_OK) return st;
    }
    return M3_OK;
}

int launch_fused_fp32_train(const m3_layer_desc& d, const m3_layer_params& p, const void* proj,
                            const float* dt_scale, void* y_out, float* h_final, float* angle,
                            float* prev_bx, void* workspace, size_t limit, hipStream_t stream) {
    const Fp32LayerParts parts = fp32_layer_parts(d, workspace);
    size_t bytes = 0;
    char* region = reinterpret_cast<char*>(fp32_layer_scratch(d, workspace, &bytes));
    const TrainRegion r = train_region(d);
    char* seg = region + r.seg;
    size_t room = r.room;
    const size_t own = al256(fp32_layer_workspace(d));
    if (fused_fp32_train_workspace(d) > own && limit > own) {  // behind the layer's workspace
        seg = reinterpret_cast<char*>(workspace) + own;
        room = limit - own;
    }
    const SegPlan sp = plan_segments(d.batch, f32k::segments(d), f32k::seg_sizes(d, false), room, false);
    return launch_fused_fp32_slice(d, p, reinterpret_cast<const float*>(proj), dt_scale,
                                   reinterpret_cast<float*>(y_out), h_final, angle, prev_bx,
                                   reinterpret_cast<float*>(region), reinterpret_cast<float*>(region + r.cn), seg,
                                   sp, stream, &parts, r.hs);
}

}  // namespace m3
