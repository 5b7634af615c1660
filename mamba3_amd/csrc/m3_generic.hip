// Generic chunked-SSD forward kernels (fp32 arithmetic, any supported shape and dtype).
//
// One workgroup owns one (batch, head) pair (the layer prefill: one block of headdim
// columns of it) and walks the sequence in chunks of `Qi` tokens, carrying the fp32 state
// (in LDS for the layer prefill, in a global buffer for chunked_ssd). Inside a chunk it
// evaluates the quadratic (L-matrix) form of the SSD
//
//   y[t,r,p] = sum_{u<=t} sum_{r'} (C~_t[r] . B~_u[r']) * M[t,u] * X_u[p,r']
//            + exp(c_t) * C~_t[r] . H[p,:]  + D * x_t[p,r]
//   M[t,u]   = exp(c_t - c_u) * (a_u + [u<t] b_u)
//   H       <- exp(c_end) * H + sum_u sum_{r'} X_u[p,r'] exp(c_end - c_u) (a_u + b_u) B~_u[r',:]
//
// which equals the reference's factored-cumsum evaluation (mamba3/ssd.py:30-65,
// 153-244) in exact arithmetic. For the layer, the trapezoid's beta term
// (mamba3/mamba3.py:212-220) is folded into the coefficients: a_u = lambda_u dt_u and
// b_u = (1 - lambda_{u+1}) dt_{u+1}, because the beta term of token u+1 uses B~_u x_u
// scaled by beta_{u+1} = (1-lambda_{u+1}) dt_{u+1} dA_{u+1}, and dA_{u+1} turns
// exp(c_t - c_{u+1}) into exp(c_t - c_u). The last token's b term hands its beta
// contribution to the next chunk through the state. For chunked_ssd's general
// two-term input (independent x_b, B_b) the B rank is doubled instead and b = 0.
//
// These kernels are the reference-shaped path for fp32 (1e-4 parity) and for shapes
// the MFMA kernels do not cover; performance is not their goal.
#include "m3_common.h"
#include "m3_kernels.h"

namespace m3 {

constexpr int kGenThreads = 1024;  // 16 waves: the loops are latency-bound
constexpr int kGenMaxLds = 64 * 1024;       // dynamic LDS without a function attribute
constexpr int kGenMaxLdsBig = 160 * 1024;   // gfx950's LDS per CU

struct GenShape {
    int B, T, H, P, N, R, Rb, G, Qi;
    int Pb, PS;  // headdim columns per workgroup and the number of column blocks (P = Pb * PS)
};

// LDS plan in floats for one workgroup.
struct GenLds {
    int tok_dt, tok_lam, c, a, bco, ec, wst, phi_run, ph, rmsB, rmsC, Cs, Bs, Xs, Sc, Ys, Hs, total;
};

// hs_lds: the (P, N) state lives in LDS with rows padded to N+1 floats.
__host__ __device__ inline GenLds gen_lds_plan(int Qi, int N, int P, int R, int Rb,
                                               bool complex_rope, bool hs_lds = false) {
    GenLds L;
    int o = 0;
    L.tok_dt = o; o += Qi + 1;
    L.tok_lam = o; o += Qi + 1;
    L.c = o; o += Qi;
    L.a = o; o += Qi;
    L.bco = o; o += Qi;
    L.ec = o; o += Qi;   // exp(c_t)
    L.wst = o; o += Qi;  // exp(c_end - c_u) (a_u + b_u): chunk-state weights
    L.phi_run = o; o += N / 2;
    L.ph = o; o += complex_rope ? Qi * (N / 2) : 0;
    L.rmsB = o; o += Qi;
    L.rmsC = o; o += Qi;
    o = (o + 3) & ~3;
    // C~ / B~ rows padded to N+1 floats: the score loop reads rows j, j+1, ... across lanes.
    L.Cs = o; o += Qi * R * (N + 1);
    L.Bs = o; o += Qi * Rb * (N + 1);
    L.Xs = o; o += Qi * Rb * P;  // P = columns of this workgroup
    L.Sc = o; o += Qi * R * Qi * Rb;
    L.Ys = o; o += Qi * R * P;
    L.Hs = o; o += hs_lds ? P * (N + 1) : 0;
    L.total = o;
    return L;
}

static int gen_pick_chunk(int N, int P, int R, int Rb, bool complex_rope, bool hs_lds = false,
                          int max_lds = kGenMaxLds) {
    for (int q = 64; q >= 1; q >>= 1) {
        if (gen_lds_plan(q, N, P, R, Rb, complex_rope, hs_lds).total * 4 <= max_lds) return q;
    }
    return 0;
}

// ---------------------------------------------------------------------------------
// Shared chunk core: scores, outputs, state update. Operates on LDS-staged tiles.
// ---------------------------------------------------------------------------------
// Hs: the (P, N) state, row p at Hs + p * hs_ld (LDS or global).
__device__ void gen_chunk_core(const GenShape& s, const GenLds& L, float* sm, float* __restrict__ Hs,
                               int hs_ld, int nvalid) {
    const int tid = threadIdx.x;
    const int Qi = s.Qi, N = s.N, P = s.Pb, R = s.R, Rb = s.Rb;  // P: this workgroup's columns
    const int rowsC = Qi * R, rowsB = Qi * Rb;
    const float* c = sm + L.c;
    const float* a = sm + L.a;
    const float* bco = sm + L.bco;
    const float* Cs = sm + L.Cs;
    const float* Bs = sm + L.Bs;
    const float* Xs = sm + L.Xs;
    float* Sc = sm + L.Sc;
    float* Ys = sm + L.Ys;
    float* ec = sm + L.ec;
    float* wst = sm + L.wst;

    // Per-token exponentials, once per chunk.
    const float c_end = c[Qi - 1];
    for (int t = tid; t < Qi; t += kGenThreads) {
        ec[t] = expf(c[t]);
        wst[t] = t < nvalid ? expf(c_end - c[t]) * (a[t] + bco[t]) : 0.f;
    }
    __syncthreads();

    // Masked, weighted scores.
    for (int idx = tid; idx < rowsC * rowsB; idx += kGenThreads) {
        const int i = idx / rowsB, j = idx % rowsB;
        const int t = i / R, u = j / Rb;
        float v = 0.f;
        if (u <= t) {
            const float* ci = Cs + i * (N + 1);
            const float* bj = Bs + j * (N + 1);
            float dot = 0.f;
            for (int n = 0; n < N; ++n) dot += ci[n] * bj[n];
            const float coef = a[u] + (u < t ? bco[u] : 0.f);
            v = dot * expf(c[t] - c[u]) * coef;
        }
        Sc[idx] = v;
    }
    __syncthreads();

    // Intra-chunk plus inter-chunk output.
    for (int idx = tid; idx < rowsC * P; idx += kGenThreads) {
        const int i = idx / P, p = idx % P;
        const int t = i / R;
        float acc = 0.f;
        const float* si = Sc + i * rowsB;
        for (int j = 0; j < (t + 1) * Rb; ++j) acc += si[j] * Xs[j * P + p];
        const float* ci = Cs + i * (N + 1);
        const float* hp = Hs + (size_t)p * hs_ld;
        float inter = 0.f;
        for (int n = 0; n < N; ++n) inter += ci[n] * hp[n];
        Ys[idx] = acc + ec[t] * inter;
    }
    __syncthreads();

    // State update.
    const float d_end = ec[Qi - 1];
    for (int idx = tid; idx < P * N; idx += kGenThreads) {
        const int p = idx / N, n = idx % N;
        float acc = 0.f;
        for (int u = 0; u < nvalid; ++u) {
            const float w = wst[u];
            float bx = 0.f;
            for (int r = 0; r < Rb; ++r) bx += Xs[(u * Rb + r) * P + p] * Bs[(u * Rb + r) * (N + 1) + n];
            acc += w * bx;
        }
        Hs[p * hs_ld + n] = d_end * Hs[p * hs_ld + n] + acc;
    }
}

// ---------------------------------------------------------------------------------
// Layer prefill from the in_proj output.
// ---------------------------------------------------------------------------------
struct GenLayerArgs {
    GenShape s;
    GenLds L;
    ProjLayout pl;
    int64_t row_stride;
    int trap, cplx;
    float eps;
    m3_layer_params prm;
    const void* proj;
    const float* dt_scale;
    void* y_out;
    float* state;      // [B,H,P,N] final state (h_final) or null
    float* angle;      // [B,H,N/2] or null
    float* prev_bx;    // [B,H,P,N] or null
};

template <typename T>
__global__ __launch_bounds__(kGenThreads) void gen_layer_prefill(GenLayerArgs A) {
    extern __shared__ float sm[];
    const GenShape& s = A.s;
    const GenLds& L = A.L;
    const int tid = threadIdx.x;
    // workgroup = (batch, head, column block): headdim columns p0 .. p0 + Pb - 1
    const int bh = blockIdx.x / s.PS, pblk = blockIdx.x % s.PS;
    const int b = bh / s.H, h = bh % s.H;
    const int g = h / (s.H / s.G);
    const int Qi = s.Qi, N = s.N, P = s.P, Pb = s.Pb, R = s.R, Nh = N / 2, NR = N * R;
    const int p0 = pblk * Pb;
    const T* proj = reinterpret_cast<const T*>(A.proj) + (int64_t)b * s.T * A.row_stride;
    T* yo = reinterpret_cast<T*>(A.y_out) + (int64_t)b * s.T * s.H * P;
    float* Hs = sm + L.Hs;  // this block's state rows, padded to N+1
    const float Ah = -expf(A.prm.A_log[h]);
    const float Dh = A.prm.D[h];
    const float dtb = A.prm.dt_bias[h];
    const float* wB = A.prm.B_norm_w;
    const float* wC = A.prm.C_norm_w;
    const float* biasB = A.prm.B_bias + (int64_t)g * NR;
    const float* biasC = A.prm.C_bias + (int64_t)g * NR;
    const float* mx = A.prm.mimo_x + (int64_t)h * P * R;
    const float* mz = A.prm.mimo_z + (int64_t)h * P * R;
    const float* md = A.prm.mimo_down + (int64_t)h * P * R;

    for (int idx = tid; idx < Pb * (N + 1); idx += kGenThreads) Hs[idx] = 0.f;
    for (int i = tid; i < Nh; i += kGenThreads) sm[L.phi_run + i] = 0.f;
    __syncthreads();

    const int nchunks = (s.T + Qi - 1) / Qi;
    for (int k = 0; k < nchunks; ++k) {
        const int s0 = k * Qi;
        const int nvalid = min(Qi, s.T - s0);
        // Token scalars for tokens s0 .. s0+Qi (one past the chunk for the trapezoid).
        for (int t = tid; t <= Qi; t += kGenThreads) {
            const int st = s0 + t;
            float dt = 0.f, lam = 1.f;
            if (st < s.T) {
                const T* row = proj + (int64_t)st * A.row_stride;
                const float sc = A.dt_scale ? A.dt_scale[((int64_t)b * s.T + st) * s.H + h] : 1.f;
                TokenGate tg = token_gate(ld_f32(row + A.pl.dt + h), dtb, sc, Ah,
                                          A.trap ? ld_f32(row + A.pl.lam + h) : 0.f, A.trap);
                dt = tg.dt;
                lam = tg.lam;
            }
            sm[L.tok_dt + t] = dt;
            sm[L.tok_lam + t] = lam;
        }
        // RMS of B and C rows of this chunk's tokens (mamba3/mamba3.py:28-35, 151-152):
        // one wave per token, lanes strided over the row, then a wave sum.
        for (int t = tid >> 6; t < Qi; t += kGenThreads / 64) {
            const int st = s0 + t;  // uniform over the wave
            float ssb = 0.f, ssc = 0.f;
            if (st < s.T) {
                const T* row = proj + (int64_t)st * A.row_stride;
                for (int e = tid & 63; e < NR; e += 64) {
                    const float vb = ld_f32(row + A.pl.B + (int64_t)g * NR + e);
                    const float vc = ld_f32(row + A.pl.C + (int64_t)g * NR + e);
                    ssb += vb * vb;
                    ssc += vc * vc;
                }
            }
            ssb = group_sum<64>(ssb);
            ssc = group_sum<64>(ssc);
            if ((tid & 63) == 0) {
                sm[L.rmsB + t] = st < s.T ? rsqrtf(ssb / NR + A.eps) : 0.f;
                sm[L.rmsC + t] = st < s.T ? rsqrtf(ssc / NR + A.eps) : 0.f;
            }
        }
        __syncthreads();
        if (tid == 0) {
            float c = 0.f;
            for (int t = 0; t < Qi; ++t) {
                const float dt = sm[L.tok_dt + t];
                c += Ah * dt;
                sm[L.c + t] = c;
                sm[L.a + t] = (A.trap ? sm[L.tok_lam + t] : 1.f) * dt;
                sm[L.bco + t] = A.trap ? (1.f - sm[L.tok_lam + t + 1]) * sm[L.tok_dt + t + 1] : 0.f;
            }
        }
        // Data-dependent RoPE angles (mamba3/mamba3.py:160-162): phi -= dt * theta. The
        // increments of all (token, pair) are read in parallel, then each pair's running
        // sum walks the chunk in LDS.
        if (A.cplx) {
            for (int idx = tid; idx < Qi * Nh; idx += kGenThreads) {
                const int t = idx / Nh, i = idx % Nh;
                const int st = s0 + t;
                sm[L.ph + idx] = st < s.T ? sm[L.tok_dt + t] * ld_f32(proj + (int64_t)st * A.row_stride + A.pl.theta + i)
                                          : 0.f;
            }
            __syncthreads();
            for (int i = tid; i < Nh; i += kGenThreads) {
                float phi = sm[L.phi_run + i];
                for (int t = 0; t < Qi; ++t) {
                    phi -= sm[L.ph + t * Nh + i];
                    sm[L.ph + t * Nh + i] = phi;
                }
                sm[L.phi_run + i] = phi;
            }
        }
        __syncthreads();
        // B~ and C~: RMSNorm * w + bias, then rotate pairs (2i, 2i+1) (mamba3/mamba3.py:38-45).
        for (int idx = tid; idx < Qi * Nh * R; idx += kGenThreads) {
            const int t = idx / (Nh * R);
            const int rem = idx % (Nh * R);
            const int i = rem / R, r = rem % R;
            const int st = s0 + t;
            float be = 0.f, bo = 0.f, ce = 0.f, co = 0.f;
            if (st < s.T) {
                const T* row = proj + (int64_t)st * A.row_stride;
                const int e0 = (2 * i) * R + r, e1 = (2 * i + 1) * R + r;
                const float rb = sm[L.rmsB + t], rc = sm[L.rmsC + t];
                be = ld_f32(row + A.pl.B + (int64_t)g * NR + e0) * rb * wB[e0] + biasB[e0];
                bo = ld_f32(row + A.pl.B + (int64_t)g * NR + e1) * rb * wB[e1] + biasB[e1];
                ce = ld_f32(row + A.pl.C + (int64_t)g * NR + e0) * rc * wC[e0] + biasC[e0];
                co = ld_f32(row + A.pl.C + (int64_t)g * NR + e1) * rc * wC[e1] + biasC[e1];
                if (A.cplx) {
                    float sn, cs;
                    sincosf(sm[L.ph + t * Nh + i], &sn, &cs);
                    const float be2 = be * cs - bo * sn, bo2 = be * sn + bo * cs;
                    const float ce2 = ce * cs - co * sn, co2 = ce * sn + co * cs;
                    be = be2; bo = bo2; ce = ce2; co = co2;
                }
            }
            float* bs = sm + L.Bs + (t * R + r) * (N + 1);
            float* cs_ = sm + L.Cs + (t * R + r) * (N + 1);
            bs[2 * i] = be;
            bs[2 * i + 1] = bo;
            cs_[2 * i] = ce;
            cs_[2 * i + 1] = co;
        }
        // MIMO x expansion (mamba3/mamba3.py:210), this block's columns.
        for (int idx = tid; idx < Qi * R * Pb; idx += kGenThreads) {
            const int t = idx / (R * Pb);
            const int r = (idx / Pb) % R, p = p0 + idx % Pb;
            const int st = s0 + t;
            float v = 0.f;
            if (st < s.T)
                v = ld_f32(proj + (int64_t)st * A.row_stride + A.pl.x + (int64_t)h * P + p) * mx[p * R + r];
            sm[L.Xs + idx] = v;
        }
        __syncthreads();

        gen_chunk_core(s, L, sm, Hs, N + 1, nvalid);

        // Gate and MIMO-down (mamba3/mamba3.py:233-238), this block's columns.
        for (int idx = tid; idx < Qi * Pb; idx += kGenThreads) {
            const int t = idx / Pb, pl = idx % Pb, p = p0 + pl;
            const int st = s0 + t;
            if (st < s.T) {
                const float z = ld_f32(proj + (int64_t)st * A.row_stride + A.pl.z + (int64_t)h * P + p);
                float out = 0.f;
                for (int r = 0; r < R; ++r) {
                    const int i = t * R + r;
                    const float y = sm[L.Ys + i * Pb + pl] + Dh * sm[L.Xs + i * Pb + pl];
                    out += md[p * R + r] * y * silu_f(z * mz[p * R + r]);
                }
                yo[((int64_t)st * s.H + h) * P + p] = cvt_out<T>(out);
            }
        }
        // prev_BX = B~_{T-1} x_{T-1}^T (mamba3/mamba3.py:247-250), this block's rows.
        if (A.prev_bx && k == nchunks - 1) {
            const int tl = nvalid - 1;
            float* pb = A.prev_bx + ((int64_t)b * s.H + h) * P * N + (int64_t)p0 * N;
            for (int idx = tid; idx < Pb * N; idx += kGenThreads) {
                const int pl = idx / N, n = idx % N;
                float v = 0.f;
                for (int r = 0; r < R; ++r)
                    v += sm[L.Bs + (tl * R + r) * (N + 1) + n] * sm[L.Xs + (tl * R + r) * Pb + pl];
                pb[idx] = v;
            }
        }
        __syncthreads();
    }
    if (A.angle && pblk == 0) {
        for (int i = tid; i < Nh; i += kGenThreads)
            A.angle[((int64_t)b * s.H + h) * Nh + i] = A.cplx ? sm[L.phi_run + i] : 0.f;
    }
    if (A.state) {
        float* hf = A.state + ((int64_t)b * s.H + h) * P * N + (int64_t)p0 * N;
        for (int idx = tid; idx < Pb * N; idx += kGenThreads) hf[idx] = Hs[(idx / N) * (N + 1) + idx % N];
    }
}

size_t generic_prefill_workspace(const m3_layer_desc&) {
    return 0;  // the running state lives in LDS
}

// The shape, headdim split and chunk of a layer under an LDS limit (Qi = 0: it does not fit).
static GenShape gen_layer_shape(const m3_layer_desc& d, int max_lds) {
    GenShape s;
    s.B = d.batch; s.T = d.seqlen; s.H = d.nheads; s.P = d.headdim; s.N = d.d_state;
    s.R = d.mimo_rank; s.Rb = d.mimo_rank; s.G = d.ngroups;
    // Split headdim over workgroups while there are idle CUs (256) and blocks keep at
    // least 16 columns: everything but the per-chunk preparation and the scores divides.
    int PS = 1;
    while (s.P % (2 * PS) == 0 && s.P / (2 * PS) >= 16 && (int64_t)d.batch * d.nheads * 2 * PS <= 256) PS *= 2;
    s.PS = PS;
    s.Pb = s.P / PS;
    s.Qi = gen_pick_chunk(s.N, s.Pb, s.R, s.Rb, d.use_complex != 0, true, max_lds);
    // A block's state rows that do not fit the LDS even at one token per chunk (d_state 512
    // with headdim 256 at large batch x heads): narrower column blocks, PS the next divisor
    // of P.
    for (int ps = PS + 1; s.Qi == 0 && ps <= s.P; ++ps) {
        if (s.P % ps != 0) continue;
        s.PS = ps;
        s.Pb = s.P / ps;
        s.Qi = gen_pick_chunk(s.N, s.Pb, s.R, s.Rb, d.use_complex != 0, true, max_lds);
    }
    return s;
}

int generic_prefill_chunk(const m3_layer_desc& d) { return gen_layer_shape(d, kGenMaxLdsBig).Qi; }

int launch_generic_prefill(const m3_layer_desc& d, const m3_layer_params& p, const void* proj,
                           const float* dt_scale, void* y_out, float* h_final, float* angle,
                           float* prev_bx, void* workspace, hipStream_t stream) {
    GenLayerArgs A;
    // Up to the CU's full LDS (one workgroup per CU): raise the kernel's dynamic-LDS limit.
    int max_lds = kGenMaxLds;
    if (d.dtype == M3_DTYPE_BF16)
        max_lds = hipFuncSetAttribute(reinterpret_cast<const void*>(&gen_layer_prefill<bf16>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, kGenMaxLdsBig) == hipSuccess
                      ? kGenMaxLdsBig : kGenMaxLds;
    else
        max_lds = hipFuncSetAttribute(reinterpret_cast<const void*>(&gen_layer_prefill<float>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, kGenMaxLdsBig) == hipSuccess
                      ? kGenMaxLdsBig : kGenMaxLds;
    A.s = gen_layer_shape(d, max_lds);
    if (A.s.Qi == 0) return M3_ERR_UNSUPPORTED;
    const int PS = A.s.PS;
    A.L = gen_lds_plan(A.s.Qi, A.s.N, A.s.Pb, A.s.R, A.s.Rb, d.use_complex != 0, true);
    A.pl = proj_layout(d);
    A.row_stride = d.proj_row_stride;
    A.trap = d.use_trapezoidal;
    A.cplx = d.use_complex;
    A.eps = d.rms_eps;
    A.prm = p;
    A.proj = proj;
    A.dt_scale = dt_scale;
    A.y_out = y_out;
    A.state = h_final;
    A.angle = angle;
    A.prev_bx = prev_bx;
    const size_t lds = (size_t)A.L.total * sizeof(float);
    const dim3 grid((unsigned)(d.batch * d.nheads * PS));
    if (d.dtype == M3_DTYPE_BF16)
        hipLaunchKernelGGL(gen_layer_prefill<bf16>, grid, dim3(kGenThreads), lds, stream, A);
    else
        hipLaunchKernelGGL(gen_layer_prefill<float>, grid, dim3(kGenThreads), lds, stream, A);
    return hipGetLastError() == hipSuccess ? M3_OK : M3_ERR_LAUNCH;
}

// ---------------------------------------------------------------------------------
// chunked_ssd on pre-processed inputs (mamba3/ssd.py:118-244).
// ---------------------------------------------------------------------------------
struct GenChunkedArgs {
    GenShape s;
    GenLds L;
    const void *x_g, *x_b, *B_g, *B_b, *C, *dt, *x_raw;
    const float *A, *D, *h_init;
    void* y;
    float* state;
};

template <typename T>
__global__ __launch_bounds__(kGenThreads) void gen_chunked(GenChunkedArgs A) {
    extern __shared__ float sm[];
    const GenShape& s = A.s;
    const GenLds& L = A.L;
    const int tid = threadIdx.x;
    const int b = blockIdx.x / s.H, h = blockIdx.x % s.H;
    const int Qi = s.Qi, N = s.N, P = s.P, R = s.R, Rb = s.Rb;
    const bool beta = A.x_b != nullptr;
    const T* xg = reinterpret_cast<const T*>(A.x_g);
    const T* xb = reinterpret_cast<const T*>(A.x_b);
    const T* Bg = reinterpret_cast<const T*>(A.B_g);
    const T* Bb = reinterpret_cast<const T*>(A.B_b);
    const T* Cc = reinterpret_cast<const T*>(A.C);
    const T* dtp = reinterpret_cast<const T*>(A.dt);
    const T* xr = reinterpret_cast<const T*>(A.x_raw);
    T* yo = reinterpret_cast<T*>(A.y);
    float* Hs = A.state + ((int64_t)b * s.H + h) * P * N;
    const float Ah = A.A[h], Dh = A.D[h];

    const float* hi = A.h_init ? A.h_init + ((int64_t)b * s.H + h) * P * N : nullptr;
    for (int idx = tid; idx < P * N; idx += kGenThreads) Hs[idx] = hi ? hi[idx] : 0.f;
    __syncthreads();

    const int nchunks = (s.T + Qi - 1) / Qi;
    for (int k = 0; k < nchunks; ++k) {
        const int s0 = k * Qi;
        const int nvalid = min(Qi, s.T - s0);
        for (int t = tid; t < Qi; t += kGenThreads) {
            const int st = s0 + t;
            sm[L.tok_dt + t] = st < s.T ? ld_f32(dtp + ((int64_t)b * s.T + st) * s.H + h) : 0.f;
        }
        // token-major (B,T,H,X,R) element (t, x, r)
        for (int idx = tid; idx < Qi * R * N; idx += kGenThreads) {
            const int t = idx / (R * N), r = (idx / N) % R, n = idx % N;
            const int st = s0 + t;
            const int64_t off = (((int64_t)b * s.T + st) * s.H + h) * N * R + (int64_t)n * R + r;
            const bool v = st < s.T;
            sm[L.Cs + (t * R + r) * (N + 1) + n] = v ? ld_f32(Cc + off) : 0.f;
            sm[L.Bs + (t * Rb + r) * (N + 1) + n] = v ? ld_f32(Bg + off) : 0.f;
            if (beta) sm[L.Bs + (t * Rb + R + r) * (N + 1) + n] = v ? ld_f32(Bb + off) : 0.f;
        }
        for (int idx = tid; idx < Qi * R * P; idx += kGenThreads) {
            const int t = idx / (R * P), r = (idx / P) % R, p = idx % P;
            const int st = s0 + t;
            const int64_t off = (((int64_t)b * s.T + st) * s.H + h) * P * R + (int64_t)p * R + r;
            const bool v = st < s.T;
            sm[L.Xs + (t * Rb + r) * P + p] = v ? ld_f32(xg + off) : 0.f;
            if (beta) sm[L.Xs + (t * Rb + R + r) * P + p] = v ? ld_f32(xb + off) : 0.f;
        }
        __syncthreads();
        if (tid == 0) {
            float c = 0.f;
            for (int t = 0; t < Qi; ++t) {
                const float dt = sm[L.tok_dt + t];
                c += Ah * dt;
                sm[L.c + t] = c;
                sm[L.a + t] = dt;
                sm[L.bco + t] = 0.f;
            }
        }
        __syncthreads();

        gen_chunk_core(s, L, sm, Hs, N, nvalid);
        __syncthreads();

        for (int idx = tid; idx < Qi * R * P; idx += kGenThreads) {
            const int t = idx / (R * P), r = (idx / P) % R, p = idx % P;
            const int st = s0 + t;
            if (st < s.T) {
                const int64_t off = (((int64_t)b * s.T + st) * s.H + h) * P * R + (int64_t)p * R + r;
                const float v = sm[L.Ys + (t * R + r) * P + p] + Dh * ld_f32(xr + off);
                yo[off] = cvt_out<T>(v);
            }
        }
        __syncthreads();
    }
}

int launch_generic_chunked(int B, int T, int H, int P, int N, int R, int dtype,
                           const void* x_g, const void* x_b, const void* B_g, const void* B_b,
                           const void* C, const void* dt, const float* A, const float* D,
                           const void* x_raw, const float* h_init, void* y, float* h_final,
                           float* state_ws, hipStream_t stream) {
    GenChunkedArgs a;
    a.s.B = B; a.s.T = T; a.s.H = H; a.s.P = P; a.s.N = N; a.s.R = R;
    a.s.Rb = x_b ? 2 * R : R;
    a.s.G = 1;
    a.s.Pb = P; a.s.PS = 1;
    // Up to the CU's full LDS when 64 KB holds less than one token per chunk (d_state 512 at
    // rank 8 with the beta terms).
    int max_lds = kGenMaxLds;
    a.s.Qi = gen_pick_chunk(N, P, R, a.s.Rb, false, false, max_lds);
    if (a.s.Qi == 0) {
        const void* f = dtype == M3_DTYPE_BF16 ? reinterpret_cast<const void*>(&gen_chunked<bf16>)
                                               : reinterpret_cast<const void*>(&gen_chunked<float>);
        if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kGenMaxLdsBig) == hipSuccess)
            max_lds = kGenMaxLdsBig;
        a.s.Qi = gen_pick_chunk(N, P, R, a.s.Rb, false, false, max_lds);
    }
    if (a.s.Qi == 0) return M3_ERR_UNSUPPORTED;
    a.L = gen_lds_plan(a.s.Qi, N, P, R, a.s.Rb, false);
    a.x_g = x_g; a.x_b = x_b; a.B_g = B_g; a.B_b = B_b; a.C = C; a.dt = dt; a.x_raw = x_raw;
    a.A = A; a.D = D; a.h_init = h_init; a.y = y;
    a.state = h_final ? h_final : state_ws;
    const size_t lds = (size_t)a.L.total * sizeof(float);
    const dim3 grid((unsigned)(B * H));
    if (dtype == M3_DTYPE_BF16)
        hipLaunchKernelGGL(gen_chunked<bf16>, grid, dim3(kGenThreads), lds, stream, a);
    else
        hipLaunchKernelGGL(gen_chunked<float>, grid, dim3(kGenThreads), lds, stream, a);
    return hipGetLastError() == hipSuccess ? M3_OK : M3_ERR_LAUNCH;
}

}  // namespace m3
