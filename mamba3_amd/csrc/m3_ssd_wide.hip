// bf16 fused chunked-SSD prefill on f16 MFMA for general layer shapes: d_state N in
// {64, 128, 256}, mimo_rank R in {1, 2, 4}, headdim P a multiple of 32 (the d_model 2048
// layer: N=256, P=128, R=4). d_state 128 / headdim 64 / rank 2 has its own kernel
// (m3_ssd_mfma.hip).
//
// Same algorithm as the other prefill kernels: the quadratic form inside a chunk and the
// state carried across chunks (mamba3/ssd.py:118-244), with the layer's preparation fused
// (mamba3/mamba3.py:197-256).
//
// Work decomposition. A workgroup owns (batch, head, PC = 32 NCG headdim columns, segment of
// the sequence) and walks its chunks of 64 (t, r) rows, Q = 64 / R tokens. PC is the whole
// headdim (128 or 64) where enough workgroups remain, so the RoPE rotation and the scores,
// which every column block of a head repeats, are done once per head. Sequences of layers whose
// heads do not fill the GPU are cut (make_plan): a state-only pass
// walks every segment but the last from a zero state in its own RoPE frame and leaves its end
// state, log-decay and angle increment, and seg_combine turns those into the state entering
// each segment.
//
// Roles. Column waves 2c and 2c + 1 own the 32 columns of group c: each keeps half of the
// state rows, H^T [n][p], in MFMA accumulators (N/32 x 2 tiles), contracts that half for all
// 64 output rows, swaps the partial sums of half the rows with the other wave through LDS and
// finishes its own rows. Helper waves (8; 4 for d_state 64) compute the scores and prepare the
// next chunk's operand tiles; workgroups of fewer column waves have extra ones for the token
// scalars and score tiles (extra_waves). Sixteen waves, four per SIMD: one wave alone issues a VALU
// instruction only every ~9 cycles, so eight waves of 256 registers (whole state rows per
// wave, no swap) left the VALU and the matrix cores idle (2.6 ms against 2.2 for both passes
// of the (2, 16384) d_model 2048 call).
//
// Bound: VALU issue and LDS bandwidth together. A chunk of that call takes a CU 12.2K cycles in
// the full pass, in which the SIMDs issue 5.1K cycles of VALU and 2.6K of MFMA and the LDS is
// busy 6.1K (profiles/pmc_segmented_prefill_kernels.md). The call (B / C normalisation 68 us,
// state pass 640, seg_combine 32, full pass 1,323) takes 2.06 ms, 0.32 of the bf16 MFMA peak;
// in blocks of 32 columns without segments (256 workgroups, every block repeating the rotation
// and the scores) it took 2.74 ms.
//
// Per chunk, in LDS (f16 unless noted):
//   C [(t,r)][n], B [(u,r')][n]       C~ / B~: normalised B^ / C^ (bc_norm_wide) rotated
//                                     by the RoPE angle; row (t,r) = t*R + r
//   XT [p][(u,r')], XwT [p][(u,r')]   x * mimo_x, and the same times the chunk weight w_u
//   S [(t,r)][(u,r')]                 masked scores (fp32 accumulated)
//   tok, part (fp32)                  token scalars; sums of dt theta of token groups
// Contractions (v_mfma_f32_16x16x32_f16, fp32 accumulation):
//   G3  Y   = diag(e^{c_t}) C~ H^T    H^T straight from the accumulators, converted to f16 in
//             registers: state tile 2s + i holds the rows n = 32 s + 8 g + 4 i + v (lane group
//             g, accumulator v), so tiles 2s and 2s + 1 give a lane the eight contraction slots
//             that its 128-bit read of a C~ row covers (the transpose reads of G4 pick the rows)
//   G4  H^T = e^{c_end} H^T + B~^T Xw    (A operand by LDS transpose reads of B~)
//   G1  S^T = B~ C~^T per causal 16x16 tile, masked by
//             Lc[t][u] = [u<=t] e^{c_t - c_u} (a_u + [u<t] b_u), plus D on the diagonal
//   G2  Y  += S X
// Output: out[t][p] = sum_r mimo_down[p,r] silu(z[t,p] mimo_z[p,r]) Y[(t,r)][p]
// (mamba3/mamba3.py:233-238). The trapezoid is folded into a_u = lambda_u dt_u and
// b_u = (1 - lambda_{u+1}) dt_{u+1}, as in the other kernels.
//
// Two phases per chunk k, a barrier after each:
//   contract  column waves G3, G4; helpers G1, chunk k+1's rotation and X rows in registers,
//             chunk k+2's token scalars
//   output    column waves G2, gate, store; helpers write chunk k+1's tiles, form chunk k+2's
//             angle sums and issue its reads
#include <algorithm>

#include "m3_common.h"
#include "m3_kernels.h"
#include "m3_mfma.h"
#include "m3_segments.h"

namespace m3 {
namespace wd {

constexpr int ROWS = 64;   // (t, r) rows per chunk
constexpr int PW = 32;     // headdim columns per column group (two waves)
constexpr int PADS = 8;    // f16 row padding of the S tile
// f16 row padding of the X^T / Xw^T tiles: a row stride of 36 32-bit words.
constexpr int PADX = 8;
// f16 row padding of the C~ / B~ tiles: a row stride of 8 (mod 16) 32-bit words keeps the
// operand and transpose reads of those tiles free of most bank conflicts.
constexpr int PADCB = 16;
constexpr float kHScale = 1.f / 256.f;  // the f16 state operand holds h * kHScale

struct Tok {
    float c2[ROWS];  // inclusive prefix of A dt over the chunk, log2 units
    float av[ROWS];  // a_u = lambda_u dt_u
    float bv[ROWS];  // b_u = (1 - lambda_{u+1}) dt_{u+1}
    float ec[ROWS];  // exp2(c2_t) / kHScale: inter-chunk output scale
    float w[ROWS];   // exp2(c2_end - c2_u) (a_u + b_u): chunk-state weight
    float dt[ROWS];  // dt_t
    float dec;       // exp2(c2_end): chunk decay of the state
};

// Column groups per workgroup: headdim in blocks of 128, 64 or 32 columns (128 columns of
// d_state 256 at rank 1, whose helper threads each prepare 16 tokens, would spill).
constexpr int max_groups(int N, int R) { return N == 256 && R == 1 ? 2 : 4; }
inline int column_groups(int P, int N, int R) {
    return std::min(max_groups(N, R), P % 128 == 0 ? 4 : P % 64 == 0 ? 2 : 1);
}

// Helper thread layout: N/4 lanes (one 4-column group, two RoPE pairs, each) share a token
// group; GR groups of TPT tokens cover the chunk.
template <int N, int R>
struct Layout {
    static constexpr int HELPERS = N == 64 ? 4 : 8;  // helper waves
    static constexpr int Q = ROWS / R;               // tokens per chunk
    static constexpr int LPT = N / 4;                // lanes per token group
    static constexpr int GR = 64 * HELPERS / LPT;
    static constexpr int TPT = Q / GR;
    static_assert(TPT >= 1 && TPT * GR == Q, "token groups cover the chunk");
};

template <int N, int R, int NCG, bool FULL>
struct __align__(16) Smem {
    static constexpr int PC = PW * NCG;
    f16 B[ROWS][N + PADCB];
    f16 C[FULL ? ROWS : 1][N + PADCB];
    f16 XT[FULL ? PC : 1][ROWS + PADX];
    f16 XwT[PC][ROWS + PADX];
    f16 S[FULL ? ROWS : 1][ROWS + PADS];
    f32x4 ex[FULL ? NCG : 1][2][2][2][64];  // partial outputs for the group's other wave: [from][row tile % 2][p tile]
    Tok tok[3];                             // by chunk mod 3
    alignas(16) float part[Layout<N, R>::GR][N / 2];     // sum of dt theta per token group
    alignas(16) float gate[FULL ? PC : 1][2][R];         // mimo_z, mimo_down * sB sC sX of the columns
    F16Scales scl;                          // operand scales of the (group, head)
};

struct Args {
    int B, T, H, G, P, PS;
    int trap, cplx;
    int64_t rs;  // proj row stride (elements)
    ProjLayout pl;
    m3_layer_params prm;
    const bf16* proj;
    const float* dt_scale;
    const f16* Bn;  // [B*T][G][N*R] pair-packed normalised B^
    const f16* Cn;
    bf16* y_out;    // [B*T][H*P]
    float* h_final;
    float* angle;
    float* prev_bx;
    // segments of the sequence (segs = 1: none), of which a launch takes lo .. hi - 1; per segment
    // but the last and pair, the state pass's end state, which seg_combine turns into the state
    // entering the next segment. The state entering segment e is kept in slot (e - 1) % slots.
    int segs, seg0;
    int lo, hi, slots;
    f32x4* hseg;  // [slot][pair block][column group][n half][tile][lane]
    float* lseg;  // log2 of the segment's decay, [seg][b h]
    float* aseg;  // its RoPE angle increment, [seg][b h][pair]
};

// v, rounded to fp32: keeps the product behind v out of a fused conversion.
__device__ __forceinline__ float opaque_f(float v) {
    asm("" : "+v"(v));
    return v;
}

__device__ __forceinline__ float readlane(float v, int l) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

// ---------------------------------------------------------------------------------
// Normalised B^ / C^ per (token, group) (mamba3/mamba3.py:19-35, 142-157): RMSNorm over
// the N*R row times the weight, plus the bias, in f16, pair-packed: the 32-bit word
// i*R + r holds (value[n=2i][r], value[n=2i+1][r]).
// ---------------------------------------------------------------------------------
constexpr int kWideBcRows = 4;  // (token, group) rows per wave of bc_norm_wide

// The 2R raw bf16 of one RoPE pair of a B / C row as R words (two elements per word, in
// order), by one vector load when the row layout allows it.
template <int R>
__device__ __forceinline__ void load_raw_pair(const bf16* p, bool vec, unsigned (&w)[R]) {
    if (vec) {
        if constexpr (R == 4) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(p);
            w[0] = v[0]; w[1] = v[1]; w[2] = v[2]; w[3] = v[3];
        } else if constexpr (R == 2) {
            const u32x2 v = *reinterpret_cast<const u32x2*>(p);
            w[0] = v[0]; w[1] = v[1];
        } else {
            w[0] = *reinterpret_cast<const unsigned*>(p);
        }
    } else {
        const unsigned short* q = reinterpret_cast<const unsigned short*>(p);
#pragma unroll
        for (int e = 0; e < R; ++e) w[e] = (unsigned)q[2 * e] | ((unsigned)q[2 * e + 1] << 16);
    }
}

// Raw element e of a pair's words, as float.
template <int R>
__device__ __forceinline__ float raw_elem(const unsigned (&w)[R], int e) {
    return __builtin_bit_cast(float, (e & 1) ? (w[e >> 1] & 0xffff0000u) : (w[e >> 1] << 16));
}

// One wave normalises kWideBcRows consecutive (token, group) rows: all their reads are
// issued first, the norm weights are read once, the biases and the operand scales once per
// distinct group of the rows (a scalar branch: a row is one wave's).
template <int N, int R>
__global__ __launch_bounds__(256) void bc_norm_wide(const bf16* __restrict__ proj, int64_t rs,
                                                    int64_t offB, int64_t offC, int G,
                                                    int64_t nrows, float eps, int vec,
                                                    const float* __restrict__ wB,
                                                    const float* __restrict__ biasB,
                                                    const float* __restrict__ wC,
                                                    const float* __restrict__ biasC,
                                                    f16* __restrict__ Bn, f16* __restrict__ Cn) {
    constexpr int NH = N / 2, NR = N * R, PPL = (NH + 63) / 64, KR = kWideBcRows;
    const int lane = threadIdx.x & 63;
    const int64_t l0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * KR;
    if (l0 >= nrows) return;
    // Lane pairs i = lane + 64 j (j < PPL); pair i covers raw elements 2iR .. 2iR+2R-1:
    // (n=2i, r) at 2iR + r, (n=2i+1, r) at 2iR + R + r. Rows past the end read the last row
    // and store nothing.
    unsigned rwb[KR][PPL][R], rwc[KR][PPL][R];
    int gg[KR];
#pragma unroll
    for (int k = 0; k < KR; ++k) {
        const int64_t tg = l0 + k < nrows ? l0 + k : nrows - 1;
        const int64_t tok = tg / G;
        gg[k] = (int)(tg % G);
        const bf16* rowB = proj + tok * rs + offB + (int64_t)gg[k] * NR;
        const bf16* rowC = proj + tok * rs + offC + (int64_t)gg[k] * NR;
#pragma unroll
        for (int j = 0; j < PPL; ++j) {
            const int i = lane + 64 * j;
            if (i < NH) {
                load_raw_pair<R>(rowB + 2 * i * R, vec, rwb[k][j]);
                load_raw_pair<R>(rowC + 2 * i * R, vec, rwc[k][j]);
            } else {
#pragma unroll
                for (int e = 0; e < R; ++e) rwb[k][j][e] = rwc[k][j][e] = 0u;
            }
        }
    }
    float wvb[PPL][2 * R], wvc[PPL][2 * R];
    float mwb = 0.f, mwc = 0.f;
#pragma unroll
    for (int j = 0; j < PPL; ++j) {
        const int i = lane + 64 * j;
#pragma unroll
        for (int e = 0; e < 2 * R; ++e) {
            wvb[j][e] = i < NH ? wB[2 * i * R + e] : 0.f;
            wvc[j][e] = i < NH ? wC[2 * i * R + e] : 0.f;
            mwb = fmaxf(mwb, fabsf(wvb[j][e]));
            mwc = fmaxf(mwc, fabsf(wvc[j][e]));
        }
    }
    mwb = wave_max(mwb);
    mwc = wave_max(mwc);
    float bvb[PPL][2 * R], bvc[PPL][2 * R];
    float ib = 1.f, ic = 1.f;
    int gcur = -1;
#pragma unroll
    for (int k = 0; k < KR; ++k) {
        const int gk = __builtin_amdgcn_readfirstlane(gg[k]);
        if (gk != gcur) {
            // biases and operand scales of the row's group (1 unless the parameters are large)
            gcur = gk;
            float mbb = 0.f, mbc = 0.f;
#pragma unroll
            for (int j = 0; j < PPL; ++j) {
                const int i = lane + 64 * j;
#pragma unroll
                for (int e = 0; e < 2 * R; ++e) {
                    bvb[j][e] = i < NH ? biasB[(int64_t)gk * NR + 2 * i * R + e] : 0.f;
                    bvc[j][e] = i < NH ? biasC[(int64_t)gk * NR + 2 * i * R + e] : 0.f;
                    mbb = fmaxf(mbb, fabsf(bvb[j][e]));
                    mbc = fmaxf(mbc, fabsf(bvc[j][e]));
                }
            }
            ib = 1.f / bc_row_scale<N, R>(mwb, wave_max(mbb));
            ic = 1.f / bc_row_scale<N, R>(mwc, wave_max(mbc));
        }
        float sb = 0.f, sc = 0.f;
#pragma unroll
        for (int j = 0; j < PPL; ++j)
#pragma unroll
            for (int e = 0; e < 2 * R; ++e) {
                const float vb = raw_elem<R>(rwb[k][j], e), vc = raw_elem<R>(rwc[k][j], e);
                sb += vb * vb;
                sc += vc * vc;
            }
        sb = lane_sum<64>(sb);
        sc = lane_sum<64>(sc);
        const float nb = rsqrtf(sb * (1.f / NR) + eps), nc = rsqrtf(sc * (1.f / NR) + eps);
        if (l0 + k >= nrows) continue;
        const int64_t tg = l0 + k;
#pragma unroll
        for (int j = 0; j < PPL; ++j) {
            const int i = lane + 64 * j;
            if (i >= NH) continue;
            // pair-packed: word r = (value[n=2i][r], value[n=2i+1][r])
            unsigned ob[R], oc[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int e0 = r, e1 = R + r;
                ob[r] = bits(f16x2{(f16)((raw_elem<R>(rwb[k][j], e0) * nb * wvb[j][e0] + bvb[j][e0]) * ib),
                                   (f16)((raw_elem<R>(rwb[k][j], e1) * nb * wvb[j][e1] + bvb[j][e1]) * ib)});
                oc[r] = bits(f16x2{(f16)((raw_elem<R>(rwc[k][j], e0) * nc * wvc[j][e0] + bvc[j][e0]) * ic),
                                   (f16)((raw_elem<R>(rwc[k][j], e1) * nc * wvc[j][e1] + bvc[j][e1]) * ic)});
            }
            f16* pb = Bn + tg * NR + 2 * i * R;
            f16* pc = Cn + tg * NR + 2 * i * R;
            if constexpr (R == 4) {
                *reinterpret_cast<u32x4*>(pb) = u32x4{ob[0], ob[1], ob[2], ob[3]};
                *reinterpret_cast<u32x4*>(pc) = u32x4{oc[0], oc[1], oc[2], oc[3]};
            } else if constexpr (R == 2) {
                *reinterpret_cast<u32x2*>(pb) = u32x2{ob[0], ob[1]};
                *reinterpret_cast<u32x2*>(pc) = u32x2{oc[0], oc[1]};
            } else {
                *reinterpret_cast<unsigned*>(pb) = ob[0];
                *reinterpret_cast<unsigned*>(pc) = oc[0];
            }
        }
    }
}

// (e, o) rotated by the angle whose (cos, sin) is kA: (e cos - o sin, e sin + o cos).
__device__ __forceinline__ unsigned rotate_pair(unsigned word, f16x2 kA, f16x2 kS) {
    const f16x2 v = as_f16x2(word);
    const f16x2 u = f16x2{v[1], v[1]} * kS;
    return bits(f16x2{v[0], v[0]} * kA + f16x2{-u[0], u[1]});
}

__device__ __forceinline__ float bf(unsigned u) { return __builtin_bit_cast(float, u << 16); }

// One of the causal score tiles (ti, ui), ui <= ti, listed row by row as 0..9. A lane's four u-rows
// 16 ui + 4 g16 + v cover NU tokens; their mask factors are read (unconditionally: every index
// is below Q) and formed before the contraction. The skip term D enters the masked scores,
// which carry 1 / (sB sC).
template <int N, int R, typename SM>
__device__ __forceinline__ void score_tile(SM& sm, const Tok& tk, int idx, int l16, int g16, float Dh) {
    constexpr int KN = N / 32;
    const int ti = idx < 1 ? 0 : idx < 3 ? 1 : idx < 6 ? 2 : 3;
    const int ui = idx - ti * (ti + 1) / 2;
    constexpr int NU = R >= 4 ? 1 : 4 / R;
    const unsigned trow = 16 * ti + l16, t = trow / R;
    const unsigned ub = (unsigned)(16 * ui + 4 * g16) / R;
    const f16* pa = &sm.B[16 * ui + l16][8 * g16];
    const f16* pb = &sm.C[16 * ti + l16][8 * g16];
    const float ct = tk.c2[t];
    float fu[NU];
#pragma unroll
    for (int j = 0; j < NU; ++j) {
        const unsigned u = ub + j;
        const float e = __builtin_amdgcn_exp2f(ct - tk.c2[u]);
        const float ab = fmaf(tk.bv[u], u < t ? 1.f : 0.f, tk.av[u]);
        fu[j] = u <= t ? e * ab : 0.f;
    }
    f32x4 sacc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KN; ++s) {
        const f16x8 A = *reinterpret_cast<const f16x8*>(pa + 32 * s);
        const f16x8 Bo = *reinterpret_cast<const f16x8*>(pb + 32 * s);
        sacc = mfma16(A, Bo, sacc);
    }
    // lane: u-row 16 ui + 4 g16 + v, t-row 16 ti + l16
    f16x4 sv;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const float val = sacc[v] * fu[v * NU / 4];
        sv[v] = (f16)(16 * ui + 4 * g16 + v == (int)trow ? val + Dh : val);
    }
    *reinterpret_cast<f16x4*>(&sm.S[trow][16 * ui + 4 * g16]) = sv;
}

// Waves beside the column and the helper waves: one computes the token scalars, the others take
// score tiles. As many as registers and the 16 waves of a workgroup leave: none beside four
// column groups of d_state 128 and 256 (helper 3 has the token scalars there) or where the
// waves would spill. With few column waves a chunk's time is that of its longest helper: of
// 6,650 cycles at d_state 128 rank 4 in one column group, the token wave's angles, scalars and
// scores took 4,100.
template <int N, int R, int NCG, bool FULL>
constexpr int extra_waves() {
    if (N != 64 && (NCG == 4 || (N == 256 && NCG == 2))) return 0;
    if (!FULL) return 1;
    if (N == 64) return R == 1 && NCG == 4 ? 0 : 4;
    return N == 256 ? 2 : NCG == 2 ? 4 : 6;
}
template <int N, int R, int NCG, bool FULL>
constexpr int kExtra = extra_waves<N, R, NCG, FULL>();
template <int N, int R, int NCG, bool FULL>
constexpr int kWaves = 2 * NCG + Layout<N, R>::HELPERS + kExtra<N, R, NCG, FULL>;

template <int N, int R, int NCG, bool FULL>
__global__ __launch_bounds__((64 * kWaves<N, R, NCG, FULL>),
                             (N == 256 ? (kWaves<N, R, NCG, FULL> + 3) / 4 : 4)) void ssd_wide(Args a) {
    using L = Layout<N, R>;
    constexpr int Q = L::Q, LPT = L::LPT, GR = L::GR, TPT = L::TPT, HELPERS = L::HELPERS;
    constexpr int CW = 2 * NCG;     // column waves
    constexpr int EXTRA = kExtra<N, R, NCG, FULL>;
    constexpr int TILERS = EXTRA > 0 ? EXTRA - 1 : 0;  // extra waves that take score tiles, two each
    constexpr int NH = N / 2;       // RoPE pairs
    constexpr int NR = N * R;
    constexpr int NT = N / 32;      // state row tiles of a wave (half of n)
    constexpr int KN = N / 32;      // k-steps over n
    constexpr int PC = PW * NCG;
    constexpr int HT = 64 * HELPERS;
    constexpr int XTH = FULL ? HT : 64 * CW;  // threads with X jobs
    constexpr int TPL = 4 / R;      // tokens per lane in an output tile
    constexpr int XT = Q * PC / XTH; // X elements per thread: consecutive tokens of one column
    __shared__ Smem<N, R, NCG, FULL> sm;

    // wave index in an SGPR, so the role branches below are scalar branches
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g16 = lane >> 4, l16 = lane & 15;
    const int npairs = a.B * a.H * a.PS;
    // Workgroups go to the 8 XCDs round-robin. Segments come longest first; within a segment the
    // (batch, head, column block) pairs are renumbered so that consecutive ones, which read the
    // same normalised B^ / C^ rows, share an XCD and its L2.
    const int so = blockIdx.x / npairs, j0 = blockIdx.x % npairs;
    const int seg = (FULL ? a.hi : min(a.hi, a.segs - 1)) - 1 - so;  // the state pass leaves the last segment out
    const int pair = (npairs % 8 == 0) ? (j0 % 8) * (npairs / 8) + j0 / 8 : j0;
    const int pblk = pair % a.PS;
    const int bh = pair / a.PS;
    const int b = bh / a.H, h = bh % a.H;
    const int grp = h / (a.H / a.G);
    const int p0 = pblk * PC;
    const int T = a.T;
    const int tbeg = (int)seg_start(seg, a.seg0);
    const int tend = seg + 1 < a.segs ? (int)seg_start(seg + 1, a.seg0) : T;
    const int nchunks = (tend - tbeg + Q - 1) / Q;
    const int64_t rs = a.rs;
    const bf16* proj = a.proj + (int64_t)b * T * rs;
    const int64_t nrs = (int64_t)a.G * NR;  // B^ / C^ token stride
    const float Ah = -expf(a.prm.A_log[h]);
    const float dtb = a.prm.dt_bias[h];
    if (wave == 0) {
        const F16Scales sc = layer_f16_scales<N, R>(a.prm, grp, h, a.P, lane);
        if (lane == 0) sm.scl = sc;
    }
    if constexpr (FULL) {
        // G2 reads 32 score columns per step: the tiles right of the diagonal in row blocks 0
        // and 2 stay zero.
        if (wave < 2) *reinterpret_cast<f16x4*>(&sm.S[32 * wave + l16][32 * wave + 16 + 4 * g16]) = f16x4{0, 0, 0, 0};
    }
    __syncthreads();
    const F16Scales scl = sm.scl.in_sgprs();
    const int hp = h * a.P + p0;  // first column of this block in x, z and y
    if constexpr (FULL) {
        for (int e = tid; e < PC * R; e += 64 * (CW + HELPERS + EXTRA)) {
            sm.gate[e / R][0][e % R] = a.prm.mimo_z[(int64_t)hp * R + e];
            sm.gate[e / R][1][e % R] = a.prm.mimo_down[(int64_t)hp * R + e] * scl.out;
        }
    }
    const int64_t sbase = (int64_t)a.B * a.H;  // (batch, head) pairs: stride of lseg / aseg

    // ---- jobs that either role runs
    // Reads of one chunk go through buffer resources that start at its first token and end at
    // the sequence's last: tokens past the end read as zero, and a lane's offset within the
    // chunk is the same for every chunk.
    auto chunk_rsrc = [&](const void* base, int kk, int64_t row_bytes) {
        const int64_t s0 = tbeg + (int64_t)kk * Q;
        return make_rsrc(reinterpret_cast<const char*>(base) + (s0 < T ? s0 * row_bytes : 0),
                         s0 < T ? (T - s0) * row_bytes : 0);
    };
    const int rb = (int)rs * 2, nb = (int)nrs * 2;  // bytes of a proj row, of a B^ / C^ token
    // X jobs: column xp, tokens xt0 .. xt0 + XT - 1
    const int xtid = FULL ? tid - 64 * CW : tid;  // helpers; column waves in the state pass
    const int xp = xtid & (PC - 1), xt0 = (xtid / PC) * XT;
    float mx[R];
#pragma unroll
    for (int r = 0; r < R; ++r) mx[r] = a.prm.mimo_x[(int64_t)(hp + xp) * R + r] * scl.inv_x;
    unsigned pxv[XT];
    const int xoff = xt0 * rb + ((int)a.pl.x + hp + xp) * 2;
    auto load_xv = [&](int kk) {
        const __amdgpu_buffer_rsrc_t r = chunk_rsrc(proj, kk, rb);
#pragma unroll
        for (int m = 0; m < XT; ++m) pxv[m] = __builtin_amdgcn_raw_buffer_load_b16(r, xoff, m * rb, kStream);
    };
    // X rows (t, r) = x_t * mimo_x[p, r] (mamba3/mamba3.py:210), and times w_t, chunk kk
    constexpr int XP = XT * R < 8 ? XT * R : 8;  // elements per stored piece
    constexpr int XV = XT * R / XP;              // pieces per thread
    static_assert(XT >= 1 && XV * XP == XT * R, "whole X pieces");
    typedef f16 xpiece __attribute__((ext_vector_type(XP)));
    xpiece xo[FULL ? XV : 1], xw[XV];
    // (The weighted product rounds to fp32 before it rounds to f16, in both passes: the compiler
    // may fuse the two into one rounding in either.)
    auto form_x = [&](int kk) {
        const Tok& tk = sm.tok[kk % 3];
#pragma unroll
        for (int m = 0; m < XT; ++m) {
            const float xval = bf(pxv[m]);
            const float w = tk.w[xt0 + m];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float v = xval * mx[r];
                if constexpr (FULL) xo[(m * R + r) / XP][(m * R + r) % XP] = (f16)v;
                xw[(m * R + r) / XP][(m * R + r) % XP] = (f16)opaque_f(v * w);
            }
        }
    };
    auto write_xw = [&]() {
#pragma unroll
        for (int v = 0; v < XV; ++v) *reinterpret_cast<xpiece*>(&sm.XwT[xp][xt0 * R + XP * v]) = xw[v];
    };
    // token scalars: lane t = token t of the chunk
    unsigned rdt0 = 0, rlam0 = 0, rdt1 = 0, rlam1 = 0;
    float sc0 = 1.f, sc1 = 1.f;
    auto load_tokens = [&](int kk) {
        const __amdgpu_buffer_rsrc_t r = chunk_rsrc(proj, kk, rb);
        const int off = (int)opaque(lane) * rb + h * 2;
        rdt0 = __builtin_amdgcn_raw_buffer_load_b16(r, off, (int)a.pl.dt * 2, 0);
        rdt1 = __builtin_amdgcn_raw_buffer_load_b16(r, off + rb, (int)a.pl.dt * 2, 0);
        if (a.trap) {
            rlam0 = __builtin_amdgcn_raw_buffer_load_b16(r, off, (int)a.pl.lam * 2, 0);
            rlam1 = __builtin_amdgcn_raw_buffer_load_b16(r, off + rb, (int)a.pl.lam * 2, 0);
        }
        if (a.dt_scale) {
            const __amdgpu_buffer_rsrc_t rd = chunk_rsrc(a.dt_scale + (int64_t)b * T * a.H, kk, (int64_t)a.H * 4);
            const int od = ((int)opaque(lane) * a.H + h) * 4;
            sc0 = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rd, od, 0, 0));
            sc1 = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rd, od + a.H * 4, 0, 0));
        }
    };
    // (No contraction, here and in the angles: the state pass and the full pass round alike.)
    auto prep_tokens = [&](int kk) {
#pragma clang fp contract(off)
        const int s0 = tbeg + kk * Q;
        const int t = lane;
        const bool v0 = t < Q && s0 + t < T, v1 = t < Q && s0 + t + 1 < T;
        // mamba3/mamba3.py:200-204, 212-216
        // computed for every lane (reads past the end are zero), then selected
        const float sp_t = fast_softplus_hw(bf(rdt0) + dtb) * sc0;
        const float sp_n = fast_softplus_hw(bf(rdt1) + dtb) * sc1;
        const float sg_t = __builtin_amdgcn_rcpf(1.f + fast_exp(-bf(rlam0)));
        const float sg_n = __builtin_amdgcn_rcpf(1.f + fast_exp(-bf(rlam1)));
        const float dt_t = v0 ? sp_t : 0.f;
        const float dt_n = v1 ? sp_n : 0.f;
        const float lam_t = v0 && a.trap ? sg_t : 1.f;
        const float lam_n = v1 && a.trap ? sg_n : 1.f;
        const float c2 = wave_incl_scan(Ah * dt_t * kLog2e);
        const float c2_end = readlane(c2, Q - 1);
        const float av = a.trap ? lam_t * dt_t : dt_t;
        const float bv = a.trap ? (1.f - lam_n) * dt_n : 0.f;
        Tok& tk = sm.tok[kk % 3];
        if (t < Q) {
            tk.dt[t] = dt_t;
            tk.c2[t] = c2;
            tk.av[t] = av;
            tk.bv[t] = bv;
            tk.ec[t] = __builtin_amdgcn_exp2f(c2) * (1.f / kHScale);
            tk.w[t] = __builtin_amdgcn_exp2f(c2_end - c2) * (av + bv);
        }
        if (t == 0) tk.dec = __builtin_amdgcn_exp2f(c2_end);
    };

    if (wave < CW) {
        // =============================== column waves ===============================
        const int cg = wave >> 1, nh = wave & 1;
        const int pw = PW * cg;      // first column of the group in the block
        const int n0 = nh * (N / 2); // first state row of the wave
        f32x4 hacc[NT][2];
#pragma unroll
        for (int t = 0; t < NT; ++t) hacc[t][0] = hacc[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (FULL && seg > 0) {
            // state entering the segment (seg_combine)
            const f32x4* hs = a.hseg + (((int64_t)((seg - 1) % a.slots) * npairs + pair) * CW + wave) * (NT * 2 * 64) + lane;
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int pt = 0; pt < 2; ++pt) hacc[t][pt] = hs[(2 * t + pt) * 64];
        }
        float ldec = 0.f;  // log2 of the segment's decay (state pass)
        // Prologue, beside the helpers' below: in the state pass the column waves form X.
        if constexpr (!FULL) load_xv(0);
        __syncthreads();  // token scalars of chunk 0 and 1
        if constexpr (!FULL) {
            form_x(0);
            write_xw();
            load_xv(1);
        }
        __syncthreads();  // angle sums of chunk 0
        __syncthreads();  // angles of chunk 0
        __syncthreads();  // tiles of chunk 0, angle sums of chunk 1

        for (int k = 0; k < nchunks; ++k) {
            const int s0 = tbeg + k * Q;
            const Tok& tk = sm.tok[k % 3];
            // ---- contract ----
            const __amdgpu_buffer_rsrc_t rp = make_rsrc(proj + (int64_t)s0 * rs, (int64_t)(T - s0) * rs * 2);
            const int zoff = ((4 * g16 / R) * (int)rs + (int)a.pl.z + hp + pw + l16) * 2;
            // The wave's half of the contraction over n for all 64 rows; row tiles 2 nh, 2 nh + 1
            // are its own to finish, the others' partial sums go to the group's other wave.
            unsigned zr_bits[FULL ? 2 : 1][2][TPL];
            f32x4 yacc[2][2];
            if constexpr (FULL) {
                f32x4 ysum[4][2];
#pragma unroll
                for (int tt = 0; tt < 4; ++tt) ysum[tt][0] = ysum[tt][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < KN / 2; ++s) {
                    f16x8 Bo[2];
#pragma unroll
                    for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            Bo[pt][v] = (f16)(hacc[2 * s][pt][v] * kHScale);
                            Bo[pt][4 + v] = (f16)(hacc[2 * s + 1][pt][v] * kHScale);
                        }
                    // row tile order: the other wave's two, then the own two; two operand rows in
                    // flight at a time (four spill the accumulators at d_state 256)
#pragma unroll
                    for (int i2 = 0; i2 < 2; ++i2) {
                        f16x8 A[2];
#pragma unroll
                        for (int i = 0; i < 2; ++i)
                            A[i] = *reinterpret_cast<const f16x8*>(&sm.C[16 * i + 32 * (i2 == 0 ? 1 - nh : nh) + l16][n0 + 32 * s + 8 * g16]);
#pragma unroll
                        for (int i = 0; i < 2; ++i)
#pragma unroll
                            for (int pt = 0; pt < 2; ++pt) ysum[2 * i2 + i][pt] = mfma16(A[i], Bo[pt], ysum[2 * i2 + i][pt]);
                        if constexpr (N == 256) M3_FENCE();
                    }
                }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int pt = 0; pt < 2; ++pt) {
                        sm.ex[cg][nh][i][pt][lane] = ysum[i][pt];
                        yacc[i][pt] = ysum[2 + i][pt];
                    }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int q = 0; q < TPL; ++q) {
                        const int so = ((32 * nh + 16 * i) / R + q) * (int)rs * 2;
                        zr_bits[i][0][q] = __builtin_amdgcn_raw_buffer_load_b16(rp, zoff, so, kStream);
                        zr_bits[i][1][q] = __builtin_amdgcn_raw_buffer_load_b16(rp, zoff + 32, so, kStream);
                    }
            }
            {
                const float dec = tk.dec;
                if constexpr (!FULL) ldec += tk.c2[Q - 1];
                f16x8 Xo[2][2];
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int pt = 0; pt < 2; ++pt)
                        Xo[s][pt] = *reinterpret_cast<const f16x8*>(&sm.XwT[pw + 16 * pt + l16][32 * s + 8 * g16]);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    hacc[t][0] *= dec;
                    hacc[t][1] *= dec;
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        const f16* bp = &sm.B[32 * s + 8 * g16 + (l16 >> 2)][n0 + 32 * (t >> 1) + 4 * (t & 1) + 8 * (l16 & 3)];
                        const f16x4 lo = ld_tr(bp);
                        const f16x4 hi = ld_tr(bp + 4 * (N + PADCB));
                        const f16x8 A = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                        hacc[t][0] = mfma16(A, Xo[s][0], hacc[t][0]);
                        hacc[t][1] = mfma16(A, Xo[s][1], hacc[t][1]);
                    }
                }
            }
            __syncthreads();
            // ---- output ----
            if constexpr (FULL) {
                // y rows of this chunk; stores past the last token fall outside and are dropped
                const __amdgpu_buffer_rsrc_t ry =
                    make_rsrc(a.y_out + ((int64_t)b * T + s0) * a.H * a.P, (int64_t)(T - s0) * a.H * a.P * 2);
                f16x8 Xo[2][2];
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int pt = 0; pt < 2; ++pt)
                        Xo[s][pt] = *reinterpret_cast<const f16x8*>(&sm.XT[pw + 16 * pt + l16][32 * s + 8 * g16]);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int tt = 2 * nh + i;  // scalar
#pragma unroll
                    for (int pt = 0; pt < 2; ++pt) yacc[i][pt] += sm.ex[cg][1 - nh][i][pt][lane];
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float e = tk.ec[(16 * tt + 4 * g16 + v) / R];
                        yacc[i][0][v] *= e;
                        yacc[i][1][v] *= e;
                    }
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        if (s > nh) break;  // columns past the row block
                        const f16x8 A = *reinterpret_cast<const f16x8*>(&sm.S[16 * tt + l16][32 * s + 8 * g16]);
                        yacc[i][0] = mfma16(A, Xo[s][0], yacc[i][0]);
                        yacc[i][1] = mfma16(A, Xo[s][1], yacc[i][1]);
                    }
#pragma unroll
                    for (int q = 0; q < TPL; ++q) {
                        const int st = (16 * tt + 4 * g16) / R + q;  // chunk token
#pragma unroll
                        for (int pt = 0; pt < 2; ++pt) {
                            const float z = bf(zr_bits[i][pt][q]);
                            float o = 0.f;
#pragma unroll
                            for (int r = 0; r < R; ++r) {
                                const float zr = z * sm.gate[pw + 16 * pt + l16][0][r];
                                o += sm.gate[pw + 16 * pt + l16][1][r] * zr * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-zr * kLog2e)) * yacc[i][pt][q * R + r];
                            }
                            __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, (bf16)o), ry,
                                                                  (st * a.H * a.P + hp + pw + 16 * pt + l16) * 2, 0, kStream);
                        }
                    }
                }
            }
            if constexpr (!FULL) {
                form_x(k + 1);
                write_xw();
                load_xv(k + 2);
            }
            __syncthreads();
        }
        if constexpr (FULL) {
            // Final state h[p][n] (fp32) from the accumulators.
            if (a.h_final && tend == T) {
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int pt = 0; pt < 2; ++pt)
                        *reinterpret_cast<f32x4*>(a.h_final + ((int64_t)bh * a.P + p0 + pw + 16 * pt + l16) * N + n0 + 32 * (t >> 1) + 8 * g16 + 4 * (t & 1)) = hacc[t][pt] * scl.state;
            }
        } else {
            f32x4* hs = a.hseg + (((int64_t)(seg % a.slots) * npairs + pair) * CW + wave) * (NT * 2 * 64) + lane;
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int pt = 0; pt < 2; ++pt) hs[(2 * t + pt) * 64] = hacc[t][pt];
            if (wave == 0 && lane == 0 && pblk == 0) a.lseg[(int64_t)seg * sbase + bh] = ldec;
        }
    } else if (EXTRA > 0 && wave >= CW + HELPERS) {
        // =============================== extra waves ===============================
        __builtin_amdgcn_s_setprio(3);
        const int ew = wave - CW - HELPERS;
        const bool token_wave = ew == TILERS;
        const float Dh = a.prm.D[h] * scl.inv_bc;
        if (token_wave) {
            load_tokens(0);
            prep_tokens(0);
            load_tokens(1);
            prep_tokens(1);
            load_tokens(2);
        }
        __syncthreads();  // token scalars of chunk 0 and 1
        __syncthreads();  // angle sums of chunk 0
        __syncthreads();  // angles of chunk 0
        __syncthreads();  // tiles of chunk 0, angle sums of chunk 1
        for (int k = 0; k < nchunks; ++k) {
            if (token_wave) {
                prep_tokens(k + 2);
                load_tokens(k + 3);
            } else if constexpr (FULL) {
#pragma unroll 1
                for (int idx = ew; idx < 2 * TILERS && idx < 10; idx += TILERS) score_tile<N, R>(sm, sm.tok[k % 3], idx, l16, g16, Dh);
            }
            __syncthreads();
            __syncthreads();
        }
    } else {
        // =============================== helper waves ===============================
        __builtin_amdgcn_s_setprio(3);  // the helpers' chains end both phases; the column waves have slack
        const int hw = wave - CW, htid = tid - 64 * CW;
        const float Dh = a.prm.D[h] * scl.inv_bc;
        const f16* Bn = a.Bn + (int64_t)b * T * nrs + (int64_t)grp * NR;
        const f16* Cn = a.Cn + (int64_t)b * T * nrs + (int64_t)grp * NR;
        // rotation jobs: RoPE pairs 2 hl, 2 hl + 1 (columns 4 hl ..) of tokens tg TPT + m
        const int hl = lane % LPT, tg = htid / LPT;
        unsigned pwb[TPT][2][R], pwc[FULL ? TPT : 1][2][R];  // raw words, loaded a chunk ahead
        const int bcoff = tg * TPT * nb + 8 * hl * R;
        auto load_words = [&](const __amdgpu_buffer_rsrc_t& r, int so, unsigned (&w)[2][R]) {
            if constexpr (R == 4) {
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, bcoff + 16 * e, so, 0);
                    w[e][0] = v[0]; w[e][1] = v[1]; w[e][2] = v[2]; w[e][3] = v[3];
                }
            } else if constexpr (R == 2) {
                const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, bcoff, so, 0);
                w[0][0] = v[0]; w[0][1] = v[1]; w[1][0] = v[2]; w[1][1] = v[3];
            } else {
                const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, bcoff, so, 0);
                w[0][0] = v[0]; w[1][0] = v[1];
            }
        };
        auto load_bc = [&](int kk) {
            const __amdgpu_buffer_rsrc_t r = chunk_rsrc(Bn, kk, nb);
#pragma unroll
            for (int m = 0; m < TPT; ++m) load_words(r, m * nb, pwb[m]);
            if constexpr (FULL) {
                const __amdgpu_buffer_rsrc_t rc = chunk_rsrc(Cn, kk, nb);
#pragma unroll
                for (int m = 0; m < TPT; ++m) load_words(rc, m * nb, pwc[m]);
            }
        };
        // theta of the rotation jobs' two pairs, raw bf16 x 2: [0] of the chunk to rotate next,
        // [1] of the one after it
        unsigned pth[2][TPT] = {};
        const bool thvec = a.rs % 2 == 0 && a.pl.theta % 2 == 0 && reinterpret_cast<uintptr_t>(a.proj) % 4 == 0;
        const int thoff = tg * TPT * rb + ((int)a.pl.theta + 2 * hl) * 2;
        auto load_theta = [&](int kk) {
            if (!a.cplx) return;  // no theta columns
            const __amdgpu_buffer_rsrc_t r = chunk_rsrc(proj, kk, rb);
            if (thvec) {
#pragma unroll
                for (int m = 0; m < TPT; ++m) pth[1][m] = __builtin_amdgcn_raw_buffer_load_b32(r, thoff, m * rb, 0);
            } else {
#pragma unroll
                for (int m = 0; m < TPT; ++m)
                    pth[1][m] = (unsigned)__builtin_amdgcn_raw_buffer_load_b16(r, thoff, m * rb, 0) |
                                ((unsigned)__builtin_amdgcn_raw_buffer_load_b16(r, thoff + 2, m * rb, 0) << 16);
            }
        };
        // this thread's sums of dt theta over its token group, chunk kk (theta in pth[1])
        auto angle_sums = [&](int kk) {
            if (!a.cplx) return;
            const Tok& tk = sm.tok[kk % 3];
            f32x2 ps = f32x2{0.f, 0.f};
#pragma unroll
            for (int m = 0; m < TPT; ++m) {
                const float dt = tk.dt[tg * TPT + m];
                ps[0] = fmaf(dt, bf(pth[1][m]), ps[0]);
                ps[1] = fmaf(dt, __builtin_bit_cast(float, pth[1][m] & 0xffff0000u), ps[1]);
            }
            *reinterpret_cast<f32x2*>(&sm.part[tg][2 * hl]) = ps;
        };
        f32x2 phi_run = f32x2{0.f, 0.f};  // pair angles at the start of the chunk to rotate next
        if (FULL && a.cplx)
#pragma unroll 4
            for (int j = 0; j < seg; ++j)
                phi_run += *reinterpret_cast<const f32x2*>(a.aseg + ((int64_t)j * sbase + bh) * NH + 2 * hl);
        // (cos, sin) of chunk kk's pairs: phi_t[i] = phi_{t-1}[i] - dt_t theta_t[i]
        // (mamba3/mamba3.py:160-162), theta in pth[0]
        f16x2 kA[TPT][2];
        auto angles = [&](int kk) {
            const Tok& tk = sm.tok[kk % 3];
            f32x2 ph = phi_run;
            if (a.cplx) {
                f32x2 run = phi_run;
#pragma unroll
                for (int g = 0; g < GR; ++g) {
                    if (g == tg) ph = run;
                    run -= *reinterpret_cast<const f32x2*>(&sm.part[g][2 * hl]);
                }
                phi_run = run;
            }
#pragma unroll
            for (int m = 0; m < TPT; ++m) {
                kA[m][0] = kA[m][1] = f16x2{(f16)1.f, (f16)0.f};
                if (a.cplx) {
                    const float dt = tk.dt[tg * TPT + m];
                    ph[0] = fmaf(-dt, bf(pth[0][m]), ph[0]);
                    ph[1] = fmaf(-dt, __builtin_bit_cast(float, pth[0][m] & 0xffff0000u), ph[1]);
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        float sn, cs;
                        fast_sincos(ph[e], sn, cs);
                        kA[m][e] = f16x2{(f16)cs, (f16)sn};
                    }
                }
            }
        };
        // C~ / B~ rows of the words in hand (words of tokens past the end are zero), and Xw^T
        auto write_tiles = [&]() {
#pragma unroll
            for (int m = 0; m < TPT; ++m) {
                const int t = tg * TPT + m;
                const f16x2 k0 = kA[m][0], k1 = kA[m][1];
                const f16x2 s0 = __builtin_shufflevector(k0, k0, 1, 0), s1 = __builtin_shufflevector(k1, k1, 1, 0);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    *reinterpret_cast<u32x2*>(&sm.B[t * R + r][4 * hl]) =
                        u32x2{rotate_pair(pwb[m][0][r], k0, s0), rotate_pair(pwb[m][1][r], k1, s1)};
                    if constexpr (FULL)
                        *reinterpret_cast<u32x2*>(&sm.C[t * R + r][4 * hl]) =
                            u32x2{rotate_pair(pwc[m][0][r], k0, s0), rotate_pair(pwc[m][1][r], k1, s1)};
                }
            }
            if constexpr (FULL) write_xw();
        };
        auto next_theta = [&]() {
#pragma unroll
            for (int m = 0; m < TPT; ++m) pth[0][m] = pth[1][m];
        };
        const bool token_wave = EXTRA == 0 && hw == 3;

        // Prologue: chunks 0 and 1's token scalars, chunk 0's tiles, chunk 1's angle sums and
        // reads (chunks past the end read as zero).
        load_bc(0);
        if constexpr (FULL) load_xv(0);
        load_theta(0);
        if (token_wave) {
            load_tokens(0);
            prep_tokens(0);
            load_tokens(1);
            prep_tokens(1);
            load_tokens(2);
        }
        __syncthreads();
        angle_sums(0);
        next_theta();
        load_theta(1);
        __syncthreads();
        angles(0);
        if constexpr (FULL) {
            form_x(0);
            load_xv(1);
        }
        __syncthreads();
        write_tiles();
        load_bc(1);
        angle_sums(1);
        next_theta();
        load_theta(2);
        __syncthreads();

        for (int k = 0; k < nchunks; ++k) {
            const bool more = k + 1 < nchunks;
            // ---- contract ----
            if constexpr (FULL) {  // G2 of the previous chunk has read its X^T
#pragma unroll
                for (int v = 0; v < XV; ++v) *reinterpret_cast<xpiece*>(&sm.XT[xp][xt0 * R + XP * v]) = xo[v];
            }
            // the next chunk's angles and X first: their reads were issued a chunk ago
            if (more) {
                angles(k + 1);
                if constexpr (FULL) {
                    form_x(k + 1);
                    load_xv(k + 2);
                }
            }
            if (token_wave) {
                prep_tokens(k + 2);
                load_tokens(k + 3);
            }
            if constexpr (FULL) {
#pragma unroll 1
                for (int idx = 2 * TILERS + hw; idx < 10; idx += HELPERS) score_tile<N, R>(sm, sm.tok[k % 3], idx, l16, g16, Dh);
            }
            __syncthreads();
            // ---- output ----
            if (more) {
                write_tiles();
                load_bc(k + 2);
                angle_sums(k + 2);
                next_theta();
                load_theta(k + 3);
            }
            __syncthreads();
        }
        // phi_run is the angle after the last chunk (rotated by the last pass)
        if constexpr (FULL) {
            if (a.angle && tend == T && pblk == 0 && htid < LPT)
                *reinterpret_cast<f32x2*>(a.angle + (int64_t)bh * NH + 2 * hl) = phi_run;
            // prev_BX = sum_r B~_{T-1}[n][r] X_{T-1}[p][r] (mamba3/mamba3.py:247-250) from the
            // last chunk's tiles.
            if (a.prev_bx && tend == T) {
                const int tl = T - 1 - tbeg - (nchunks - 1) * Q;
                for (int idx = htid; idx < PC * N; idx += HT) {
                    const int p = idx / N, n = idx % N;
                    float v = 0.f;
#pragma unroll
                    for (int r = 0; r < R; ++r) v += (float)sm.B[tl * R + r][n] * (float)sm.XT[p][tl * R + r];
                    a.prev_bx[((int64_t)bh * a.P + p0 + p) * N + n] = v * scl.state;
                }
            }
        } else {
            if (pblk == 0 && htid < LPT)
                *reinterpret_cast<f32x2*>(a.aseg + ((int64_t)seg * sbase + bh) * NH + 2 * hl) = phi_run;
        }
    }
}

// Turns the segments' end states (from a zero start, each in its own RoPE frame, whose zero is
// its first token's incoming angle) into the states entering the next segments, in place: one
// thread per four state rows of a column, walking the segments in order. HBM-bound (two passes
// over the states); the full pass would otherwise read every earlier segment's.
template <int N, int NCG>
__global__ __launch_bounds__(256) void seg_combine(Args a) {
    constexpr int NT = N / 32, CW = 2 * NCG;
    constexpr int PER = CW * NT * 2 * 64;  // entries per pair block
    const int npairs = a.B * a.H * a.PS;
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= (int64_t)npairs * PER) return;
    const int bh = (int)(e / PER) / a.PS;
    const int w = (int)(e % PER) / (NT * 2 * 64), t = (int)(e % (NT * 2 * 64)) / 128, g16 = (int)(e % 64) / 16;
    const int i = ((w & 1) * (N / 2) + 32 * (t >> 1) + 8 * g16 + 4 * (t & 1)) / 2;  // first RoPE pair
    const int64_t sbase = (int64_t)a.B * a.H;
    auto slot = [&](int j) { return a.hseg + (int64_t)(j % a.slots) * npairs * PER + e; };
    auto angle_inc = [&](int j) {
        return *reinterpret_cast<const f32x2*>(a.aseg + ((int64_t)j * sbase + bh) * (N / 2) + i);
    };
    f32x4 h = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x2 phi = f32x2{0.f, 0.f};
    if (a.lo > 0) h = *slot(a.lo - 1);
    for (int j = 0; j < a.lo; ++j) phi += angle_inc(j);
    const int hi = min(a.hi, a.segs - 1);
#pragma unroll 2
    for (int j = a.lo; j < hi; ++j) {
        f32x4* hj = slot(j);
        const f32x4 v = *hj;
        const f32x2 inc = angle_inc(j);
        const float dec = __builtin_amdgcn_exp2f(a.lseg[(int64_t)j * sbase + bh]);
        float s0, c0, s1, c1;
        fast_sincos(phi[0], s0, c0);
        fast_sincos(phi[1], s1, c1);
        // (the first segment's state is in the sequence's frame already)
        h = j == 0 ? v : h * dec + f32x4{v[0] * c0 - v[1] * s0, v[0] * s0 + v[1] * c0,
                                         v[2] * c1 - v[3] * s1, v[2] * s1 + v[3] * c1};
        *hj = h;
        phi += inc;
    }
}

// The segments in groups of `group` (all of them, unless the workspace holds fewer states).
template <int N, int R, int NCG>
void launch_ssd(Args a, int group, hipStream_t stream) {
    const unsigned npairs = (unsigned)(a.B * a.H * a.PS);
    for (a.lo = 0; a.lo < a.segs; a.lo = a.hi) {
        a.hi = std::min(a.segs, a.lo + group);
        const int ns = std::min(a.hi, a.segs - 1) - a.lo;
        if (ns > 0) {
            hipLaunchKernelGGL((ssd_wide<N, R, NCG, false>), dim3(npairs * ns), dim3(64 * kWaves<N, R, NCG, false>), 0, stream, a);
            hipLaunchKernelGGL((seg_combine<N, NCG>), dim3((unsigned)(((int64_t)npairs * PW * NCG * N / 4 + 255) / 256)),
                               dim3(256), 0, stream, a);
        }
        hipLaunchKernelGGL((ssd_wide<N, R, NCG, true>), dim3(npairs * (a.hi - a.lo)), dim3(64 * kWaves<N, R, NCG, true>), 0, stream, a);
    }
}

// The cuts of a sequence depend on nothing but its layer and its tokens: not on the batch, so
// that a sequence gives the same bits alone and in any batch, nor on the workspace (but see
// plan_segments), nor, as they lie at fixed tokens, on the length, so that a prefix gives the same
// bits too. They are closer at the start, so that a short prompt splits finely and a long one
// into few states. Layers of 96 or more column blocks (heads times headdim / 128, 64 or 32) are
// not cut: a segmented walk does 1.5x the work (its state pass) and repeats its prologue. us per
// call, cut / uncut, one sequence of 2,048 and 4,096 tokens, d_state 64 headdim 64 rank 2: 8
// heads 75 / 135 and 110 / 258, 96 122 / 139 and 207 / 260, 128 150 / 140 and 265 / 261, 190 213 /
// 157 and 387 / 297; d_state 256 headdim 128 rank 4: 32 heads 236 / 372 and 513 / 716, 64 314 /
// 385 and 574 / 737, 96 569 / 441 and 802 / 847, 128 584 / 449 and 969 / 859. Batches of the
// 32-head layer: (1, 16384) 1,030 / 2,789, (2, 16384) 2,072 / 2,956, but (8, 2048) 1,068 / 656.
// The first cut is free, as the state at it is the walk's own: up to two segments a sequence
// is walked in one piece with the same bits ((1, 600) of that layer 132 us, 199 cut).
struct Plan : SegPlan {
    int seg0;
    int ncg;  // column groups per workgroup
};

Plan make_plan(const m3_layer_desc& d, size_t limit) {
    Plan p;
    p.ncg = column_groups(d.headdim, d.d_state, d.mimo_rank);
    const int64_t blocks = d.headdim / (PW * p.ncg);
    p.seg0 = std::max(256, d.headdim * d.d_state / 64);
    const int segs = d.nheads * blocks < 96 ? seg_count(d.seqlen, p.seg0) : 1;
    const SegSizes z = {(size_t)d.seqlen * d.ngroups * d.d_state * d.mimo_rank * sizeof(f16),
                        (size_t)d.nheads * d.headdim * d.d_state * sizeof(float),
                        d.nheads * sizeof(float), d.nheads * (d.d_state / 2) * sizeof(float)};
    static_cast<SegPlan&>(p) = plan_segments(d.batch, segs, z, limit, true);
    // Narrower blocks where they still run at once, one a CU: they repeat the rotation and the
    // scores, but each walks its chunks faster (same bits: a column's arithmetic does not depend
    // on its block). us per call in blocks of 128 / 64 / 32 columns, d_state 256 rank 4, headdim
    // 128, 32 heads, 600 tokens: one sequence 202 / 150 / 134, two 202 / 151 / 134, four 205 / 156
    // / 263, five 207 / 303 / 391; d_state 128 rank 4, headdim 64, 24 heads, 300 tokens: four
    // - / 61 / 58, six - / 62 / 112.
    const int64_t bh = (int64_t)p.batch * d.nheads * p.group;
    while (p.ncg > 1 && 2 * bh * (d.headdim / (PW * p.ncg)) <= 256) p.ncg /= 2;
    return p;
}

// One slice of the batch.
template <int N, int R>
int launch_slice(const m3_layer_desc& d, const Plan& plan, const m3_layer_params& p, const bf16* proj,
                 const float* dt_scale, bf16* y_out, float* h_final, float* angle, float* prev_bx,
                 void* workspace, hipStream_t stream) {
    const int ncg = plan.ncg;
    char* ws = reinterpret_cast<char*>(workspace);
    Args a;
    a.B = d.batch; a.T = d.seqlen; a.H = d.nheads; a.G = d.ngroups; a.P = d.headdim;
    a.PS = d.headdim / (PW * ncg);
    a.trap = d.use_trapezoidal; a.cplx = d.use_complex;
    a.rs = d.proj_row_stride;
    a.pl = proj_layout(d);
    a.prm = p;
    a.proj = proj;
    a.dt_scale = dt_scale;
    const int64_t nrows = (int64_t)d.batch * d.seqlen * d.ngroups;
    f16* bn = reinterpret_cast<f16*>(ws);
    f16* cn = reinterpret_cast<f16*>(ws + plan.rows);
    a.Bn = bn;
    a.Cn = cn;
    a.y_out = y_out;
    a.h_final = h_final;
    a.angle = angle;
    a.prev_bx = prev_bx;
    a.segs = plan.segs;
    a.seg0 = plan.seg0;
    a.slots = plan.slots;
    a.hseg = reinterpret_cast<f32x4*>(ws + plan.hseg);
    a.lseg = reinterpret_cast<float*>(ws + plan.lseg);
    a.aseg = reinterpret_cast<float*>(ws + plan.aseg);
    // vector loads of a pair's 2R raw values when every row offset keeps them aligned
    const int vec = a.rs % (2 * R) == 0 && a.pl.B % (2 * R) == 0 && a.pl.C % (2 * R) == 0 &&
                    reinterpret_cast<uintptr_t>(proj) % (4 * R) == 0;
    constexpr int rows_per_block = 4 * kWideBcRows;
    hipLaunchKernelGGL((bc_norm_wide<N, R>), dim3((unsigned)((nrows + rows_per_block - 1) / rows_per_block)),
                       dim3(256), 0, stream, a.proj, a.rs, a.pl.B, a.pl.C, a.G, nrows, d.rms_eps, vec,
                       p.B_norm_w, p.B_bias, p.C_norm_w, p.C_bias, bn, cn);
    if constexpr (max_groups(N, R) == 4) {
        if (ncg == 4) {
            launch_ssd<N, R, 4>(a, plan.group, stream);
            return hipGetLastError() == hipSuccess ? M3_OK : M3_ERR_LAUNCH;
        }
    }
    if (ncg == 2) launch_ssd<N, R, 2>(a, plan.group, stream);
    else launch_ssd<N, R, 1>(a, plan.group, stream);
    return hipGetLastError() == hipSuccess ? M3_OK : M3_ERR_LAUNCH;
}

template <int N, int R>
int launch(const m3_layer_desc& d, const m3_layer_params& p, const void* proj,
           const float* dt_scale, void* y_out, float* h_final, float* angle, float* prev_bx,
           void* workspace, size_t limit, hipStream_t stream) {
    const Plan plan = make_plan(d, limit);
    const int64_t T = d.seqlen, H = d.nheads, PN = (int64_t)d.headdim * d.d_state;
    for (int b = 0; b < d.batch; b += plan.batch) {
        m3_layer_desc part = d;
        part.batch = std::min(plan.batch, d.batch - b);
        auto at = [&](auto* q, int64_t per_row) { return q ? q + b * per_row : nullptr; };
        const int st = launch_slice<N, R>(part, plan, p, reinterpret_cast<const bf16*>(proj) + b * T * d.proj_row_stride,
                                          at(dt_scale, T * H), reinterpret_cast<bf16*>(y_out) + b * T * H * d.headdim,
                                          at(h_final, H * PN), at(angle, H * (d.d_state / 2)),
                                          at(prev_bx, H * PN), workspace, stream);
        if (st != M3_OK) return st;
    }
    return M3_OK;
}

}  // namespace wd

bool wide_prefill_supported(const m3_layer_desc& d) {
    if (d.dtype != M3_DTYPE_BF16) return false;
    if (d.headdim % wd::PW != 0) return false;
    const int N = d.d_state, R = d.mimo_rank;
    if (N != 64 && N != 128 && N != 256) return false;
    if (R != 1 && R != 2 && R != 4) return false;
    // a chunk's rows (up to 64 tokens) are addressed with 32-bit byte offsets
    const int64_t lim = (int64_t)1 << 23;
    return d.proj_row_stride < lim && (int64_t)d.ngroups * N * R < lim && (int64_t)d.nheads * d.headdim < lim;
}

size_t wide_prefill_workspace(const m3_layer_desc& d) { return wd::make_plan(d, SIZE_MAX).total; }

size_t wide_prefill_min_workspace(const m3_layer_desc& d) { return wd::make_plan(d, 0).total; }

int launch_wide_prefill(const m3_layer_desc& d, const m3_layer_params& p, const void* proj,
                        const float* dt_scale, void* y_out, float* h_final, float* angle,
                        float* prev_bx, void* workspace, size_t limit, hipStream_t stream) {
#define M3_WIDE_CASE(n, r)                                                                      \
    if (d.d_state == n && d.mimo_rank == r)                                                     \
        return wd::launch<n, r>(d, p, proj, dt_scale, y_out, h_final, angle, prev_bx, workspace, \
                                limit, stream);
    M3_WIDE_CASE(64, 1) M3_WIDE_CASE(64, 2) M3_WIDE_CASE(64, 4)
    M3_WIDE_CASE(128, 1) M3_WIDE_CASE(128, 2) M3_WIDE_CASE(128, 4)
    M3_WIDE_CASE(256, 1) M3_WIDE_CASE(256, 2) M3_WIDE_CASE(256, 4)
#undef M3_WIDE_CASE
    return M3_ERR_UNSUPPORTED;
}

}  // namespace m3
