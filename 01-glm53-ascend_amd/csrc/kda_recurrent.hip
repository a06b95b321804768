// kda_recurrent.hip -- fused recurrent KDA (delta rule with per-channel decay)
// over packed varlen sequences, for gfx950.
//
// Semantics follow the reference recurrence (bench/kda_chunk/kda_python.py:
// 253-307; device version sgl-glm53-ascend-ops/csrc/kda/recurrent/
// kda_varlen_recurrent_decode_h32.cpp:289-724): per (sequence, head) with
// state S[k][v] and per token t
//     S   <- exp(g_t)[k] * S
//     d_v  = beta_t * (v_t[v] - sum_k kn_t[k] S[k][v])
//     S   <- S + kn_t[k] d_v
//     o_v  = sum_k qn_t[k] S[k][v]           (readout after the update)
// with slot 0 the zero/padding state, per-step checkpoints and prefix
// tracking as described in kda_abi.h.
//
// MI355X mapping. The update never mixes value rows, so the state splits into
// independent rows S[:, v], each a contiguous 4*D-byte line of the
// K-contiguous pool. A row is spread over L lanes (a row group); each lane
// owns E = D/L of its K elements as E/4 16-byte vectors at K offsets
// 4*kc + 4*L*j, so every wave-wide 16-byte load covers whole 4*L-element
// segments of its rows -- complete cache lines. A lane holds the same K
// elements of NP rows. The two K-reductions per token
// (prediction and readout) are group sums over the L lanes (DPP, plus one
// ds_swizzle when L = 32), so the state tile lives in VGPRs from the first
// load to the single in-place write-back: HBM sees each state byte exactly
// once in and once out. A workgroup (4 waves) covers 4*(64/L)*NP value rows
// of one (sequence, head). The host picks the kernel and shape from the
// tokens per sequence: one token (decode) uses 32-lane rows with few rows per
// lane, so the launch has many small workgroups to stream the state; more
// (verify, prefill) run in blocks of tokens prepared once per workgroup, on
// 16-lane rows, whose reductions take four DPP steps instead of five plus an
// LDS swizzle.

#include <hip/hip_runtime.h>

#include <type_traits>

#include "kda_abi.h"
#include "kda_device.h"

namespace kda {
namespace {

constexpr int kThreads = 256;

using RecurrentLaunch = Launch<KdaRecurrentArgs>;

// A request's bounds and slot, needed at once: loaded in one round trip. (Left to
// itself the compiler moves the bounds' loads behind the slot's wait and its
// branches, a round trip more, which one-token launches of 3 us feel: 1 x 1
// tokens, H=4, log gates: 2.98 us against 3.05.)
__device__ __forceinline__ void together(int2 ends, int slot) {
    asm volatile("" ::"s"(ends.x), "s"(ends.y), "s"(slot));
}

// e^x as one v_exp_f32 of x*log2(e). The product's rounding puts the
// relative error near |x| * 2^-24 plus the instruction's own ~1 ulp; a
// result below the fp32 normal range may flush to zero.
__device__ __forceinline__ float fexp(float x) {
    return __builtin_amdgcn_exp2f(x * 1.4426950408889634f);
}

// Four consecutive K elements as loaded: 8 bytes of bf16 or 16 of fp32,
// widened to fp32 at use.
template <typename T> struct Raw4;
template <> struct Raw4<uint16_t> {
    uint2 r;
    __device__ __forceinline__ void load(const uint16_t *p) {
        r = *reinterpret_cast<const uint2 *>(p);
    }
    __device__ __forceinline__ float4 get() const {
        return make_float4(__uint_as_float(r.x << 16), __uint_as_float(r.x & 0xffff0000u),
                           __uint_as_float(r.y << 16), __uint_as_float(r.y & 0xffff0000u));
    }
};
template <> struct Raw4<float> {
    float4 r;
    __device__ __forceinline__ void load(const float *p) { r = *reinterpret_cast<const float4 *>(p); }
    __device__ __forceinline__ float4 get() const { return r; }
};

// NP values of one v row, RS elements apart, as loaded (widened at use, so
// the load is not waited for until the value is needed). Consecutive values
// (RS = 1) arrive in 16-byte or smaller vectors from addresses aligned for them
// (load) and one element per load from others (load_each; the caller looks at the
// alignment): bf16 pairs packed in words, fp32 as is. Spread ones always arrive one
// element per load.
template <typename T, int NP, int RS> struct RowIn;
template <int NP, int RS> struct RowIn<uint16_t, NP, RS> {
    static constexpr int W = RS == 1 ? NP / 2 : NP;
    static_assert(RS != 1 || NP % 2 == 0, "bf16 pairs");
    uint32_t w[W];
    __device__ __forceinline__ void load(const uint16_t *p) {
        if constexpr (RS != 1) {
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                w[i] = p[RS * i];
            }
        } else if constexpr (NP == 2) {
            w[0] = *reinterpret_cast<const uint32_t *>(p);
        } else if constexpr (NP == 4) {
            const uint2 u = *reinterpret_cast<const uint2 *>(p);
            w[0] = u.x;
            w[1] = u.y;
        } else {
#pragma unroll
            for (int i = 0; i < NP / 8; ++i) {
                const uint4 u = reinterpret_cast<const uint4 *>(p)[i];
                w[4 * i + 0] = u.x;
                w[4 * i + 1] = u.y;
                w[4 * i + 2] = u.z;
                w[4 * i + 3] = u.w;
            }
        }
    }
    // the same from an address of any alignment
    __device__ __forceinline__ void load_each(const uint16_t *p) {
        if constexpr (RS != 1) {
            load(p);
        } else {
#pragma unroll
            for (int i = 0; i < W; ++i) {
                w[i] = static_cast<uint32_t>(p[2 * i]) | (static_cast<uint32_t>(p[2 * i + 1]) << 16);
            }
        }
    }
    __device__ __forceinline__ float get(int i) const {
        if constexpr (RS != 1) {
            return __uint_as_float(w[i] << 16);
        } else {
            return __uint_as_float((i & 1) ? (w[i >> 1] & 0xffff0000u) : (w[i >> 1] << 16));
        }
    }
};
template <int NP, int RS> struct RowIn<float, NP, RS> {
    static_assert(RS != 1 || NP % 4 == 0 || NP == 2, "whole vectors");
    float x[NP];
    __device__ __forceinline__ void load(const float *p) {
        if constexpr (RS != 1) {
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                x[i] = p[RS * i];
            }
        } else if constexpr (NP == 2) {
            const float2 u = *reinterpret_cast<const float2 *>(p);
            x[0] = u.x;
            x[1] = u.y;
        } else {
#pragma unroll
            for (int i = 0; i < NP / 4; ++i) {
                const float4 u = reinterpret_cast<const float4 *>(p)[i];
                x[4 * i + 0] = u.x;
                x[4 * i + 1] = u.y;
                x[4 * i + 2] = u.z;
                x[4 * i + 3] = u.w;
            }
        }
    }
    __device__ __forceinline__ void load_each(const float *p) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            x[i] = p[RS * i];
        }
    }
    __device__ __forceinline__ float get(int i) const { return x[i]; }
};

// NP output values of one row, RS elements apart: consecutive ones (RS = 1) this
// lane's own, written as vectors to an address aligned for them; spread ones held
// alike by the row group's lanes kc, value i written by lane i.
template <typename T, int NP, int RS>
__device__ __forceinline__ void store_row(T *p, const float (&x)[NP], int kc) {
    if constexpr (RS == 1) {
        if constexpr (sizeof(T) == 2) {
            static_assert(NP % 2 == 0, "bf16 pairs");
            uint32_t w[NP / 2];
#pragma unroll
            for (int i = 0; i < NP / 2; ++i) {
                w[i] = pack_bf16x2(x[2 * i], x[2 * i + 1]);
            }
            if constexpr (NP == 2) {
                *reinterpret_cast<uint32_t *>(p) = w[0];
            } else if constexpr (NP == 4) {
                *reinterpret_cast<uint2 *>(p) = make_uint2(w[0], w[1]);
            } else {
#pragma unroll
                for (int i = 0; i < NP / 8; ++i) {
                    reinterpret_cast<uint4 *>(p)[i] =
                        make_uint4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
                }
            }
        } else if constexpr (NP == 2) {
            *reinterpret_cast<float2 *>(p) = make_float2(x[0], x[1]);
        } else {
            static_assert(NP % 4 == 0, "whole float4 vectors");
#pragma unroll
            for (int i = 0; i < NP / 4; ++i) {
                reinterpret_cast<float4 *>(p)[i] =
                    make_float4(x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]);
            }
        }
    } else {
        float mine = 0.f;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            mine = (kc == i) ? x[i] : mine;
        }
        if (kc < NP) {
            store1(p + RS * kc, mine);
        }
    }
}

template <int D, int L, int NP, typename TQK, typename TV, int GATE>
__global__ __launch_bounds__(kThreads) void recurrent_kernel(const RecurrentLaunch a) {
    constexpr int E = D / L;           // K elements per lane
    constexpr int EV = E / 4;          // 16-byte vectors per lane and row
    constexpr int RPW = 64 / L;        // row groups per wave
    constexpr int RPP = 4 * RPW;       // row groups per workgroup
    constexpr int RB = RPP * NP;       // rows per workgroup
    // A lane's NP rows are RPP apart: each wave-wide state load covers RPW
    // adjacent rows, one contiguous span.
    constexpr int RS = RPP;
    constexpr int VT = D / RB;         // workgroups per (sequence, head)
    static_assert(E % 4 == 0 && D % RB == 0, "whole vectors and whole row tiles");

    const int H = a.num_heads;
    const int HC = a.head_count;  // heads in this launch, resolved by the host
    // XCD-aware order: consecutive workgroups go to different XCDs (each with
    // its own L2), so the VT row tiles of one (sequence, head), which read the
    // same token rows, are numbered 8 apart and share an XCD.
    const int b = blockIdx.x;
    const int rest = b >> 3;
    const int vt = VT == 1 ? 0 : rest % VT;
    const int pair = VT == 1 ? b : (rest / VT) * 8 + (b & 7);
    const int n = pair / HC;
    const int head = a.head_begin + (pair - n * HC);
    if (n >= a.num_seqs) {
        return;
    }
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int kc = lane % L;
    const int rgw = wave * RPW + lane / L;  // row group in the workgroup
    const int row0 = vt * RB + rgw;  // rows row0 + RS*p, p < NP
    const int T = a.num_tokens;

    const int2 ends = a.cu_pair(n);
    int slot = a.slot_index(n);
    together(ends, slot);
    int bos = ends.x;
    int eos = ends.y;
    bos = bos < 0 ? 0 : (bos > T ? T : bos);
    eos = eos < bos ? bos : (eos > T ? T : eos);
    if (slot < 0 || static_cast<int64_t>(slot) >= a.num_slots) {
        slot = 0;
    }

    // Offset of this lane's vector j within a row of D elements.
    auto koff = [&](int j) { return 4 * kc + 4 * L * j; };
    const int64_t head_off = static_cast<int64_t>(head) * a.state_stride_head;
    // A [K,V]-contiguous pool (state_v_contiguous, the prepared_recurrent
    // layout of the reference; DECAY mode only, the launcher rejects it
    // otherwise, so the other modes compile without it) is read and written
    // in place element by element: element (k, v) of a slot and head sits at
    // k*D + v.
    const bool vpool = GATE == KDA_GATE_DECAY && a.state_v_contiguous != 0;
    float4 S[NP][EV];
    if (slot > 0) {
        const float *src = a.state + slot * a.state_stride_slot + head_off;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
#pragma unroll
            for (int j = 0; j < EV; ++j) {
                if (vpool) {
                    const float *e = src + static_cast<int64_t>(koff(j)) * D + row0 + RS * p;
                    S[p][j] = make_float4(e[0], e[D], e[2 * D], e[3 * D]);
                } else {
                    S[p][j] = load4_stream(src + static_cast<int64_t>(row0 + RS * p) * D + koff(j));
                }
            }
        }
    } else {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
#pragma unroll
            for (int j = 0; j < EV; ++j) {
                S[p][j] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
    }

    // Prefix tracking: the destination slot and the local step after which to
    // store (0 = the initial state, stored right away).
    int track_slot = 0;
    int track_len = -1;
    if (a.track_indices != nullptr) {
        track_slot = a.track_index(n);
        if (track_slot <= 0 || static_cast<int64_t>(track_slot) >= a.num_slots) {
            track_slot = 0;
        } else {
            track_len = a.track_length(n);
        }
    }
    // State tiles are touched once per launch: streamed with nontemporal
    // loads and stores so they do not evict the token rows from the caches
    // (measured ~10% more HBM throughput than cached accesses).
    auto store_state = [&](float *dst, bool vlayout) {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
#pragma unroll
            for (int j = 0; j < EV; ++j) {
                if (vlayout) {
                    float *e = dst + static_cast<int64_t>(koff(j)) * D + row0 + RS * p;
                    e[0] = S[p][j].x;
                    e[D] = S[p][j].y;
                    e[2 * D] = S[p][j].z;
                    e[3 * D] = S[p][j].w;
                } else {
                    store4_stream(dst + static_cast<int64_t>(row0 + RS * p) * D + koff(j), S[p][j]);
                }
            }
        }
    };
    if (track_slot > 0 && track_len == 0) {
        store_state(a.state + track_slot * a.state_stride_slot + head_off, vpool);
    }

    // Per-head gate constants (RAW): exp(A_log[h]) and this lane's dt_bias.
    float expA = 0.f;
    float4 dtb[EV];
#pragma unroll
    for (int j = 0; j < EV; ++j) {
        dtb[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    if constexpr (GATE == KDA_GATE_RAW) {
        expA = expf(a.A_log[head]);
#pragma unroll
        for (int j = 0; j < EV; ++j) {
            dtb[j] = load4(a.dt_bias + static_cast<int64_t>(head) * D + koff(j));
        }
    }
    const bool norm = (GATE == KDA_GATE_RAW) || (a.qk_l2norm != 0);
    const bool save_mid = a.intermediate != nullptr && slot > 0 && n < a.mid_rows;

    const TQK *qp = static_cast<const TQK *>(a.q);
    const TQK *kp = static_cast<const TQK *>(a.k);
    const TV *vp = static_cast<const TV *>(a.v);
    TV *op = static_cast<TV *>(a.out);
    using TG = typename std::conditional<GATE == KDA_GATE_RAW, uint16_t, float>::type;
    const TG *gp = static_cast<const TG *>(a.gate);

    // One token's inputs, as loaded; widened and transformed before its
    // step. The next token's are loaded while the current one computes: a
    // multi-token sequence (verify, prefill) would otherwise wait a full load
    // latency per token.
    struct TokenIn {
        Raw4<TQK> q[EV], k[EV];
        Raw4<TG> g[EV];
        RowIn<TV, NP, RS> v;
        float b;
    };
    auto fetch = [&](int t, TokenIn &in) {
        const int64_t base = (static_cast<int64_t>(t) * H + head) * D;
#pragma unroll
        for (int j = 0; j < EV; ++j) {
            in.q[j].load(qp + base + koff(j));
            in.k[j].load(kp + base + koff(j));
            in.g[j].load(gp + base + koff(j));
        }
        in.v.load(vp + base + row0);
        const int64_t bi = static_cast<int64_t>(t) * H + head;
        if constexpr (GATE == KDA_GATE_RAW) {
            in.b = bf16_to_f32(static_cast<const uint16_t *>(a.beta)[bi]);
        } else {
            in.b = static_cast<const float *>(a.beta)[bi];
        }
    };
    // A token ready for the update: scaled q, normalized k, decay, beta, v.
    struct Token {
        float4 q[EV], k[EV], dec[EV];
        float beta;
        float v[NP];
    };
    // Every row group of a workgroup needs the same per-channel decays, beta
    // and norms of a token. With one vector per lane and row (EV == 1: the
    // row groups' L lanes cover the D channels four apiece) the workgroup
    // computes them once and shares them through LDS: the row groups of the waves before kNormWave each take one
    // component of their lanes' vectors (rows groups 0-3: channels 4 kc + r),
    // wave kNormWave forms the q norm (its even row groups) and the k norm
    // (odd ones) with the same group sums every row group would use, and the
    // next wave forms beta. Each value is the same expression of the same
    // inputs as in the per-lane form, so the results are bitwise those of
    // every row group computing everything itself; the raw decode's prologue
    // (two expf and a division per channel) then runs once per (token,
    // channel) in the workgroup instead of once per row group (8x fewer).
    // Tokens alternate between two LDS sets, so one barrier per token
    // separates the writes of token t + 2 from the reads of token t.
    constexpr bool kShare = GATE != KDA_GATE_DECAY && EV == 1;
    constexpr int kNormWave = 4 / RPW;
    static_assert(!kShare || (4 * L == D && kNormWave + 1 < 4), "roles of the shared prologue");
    __shared__ float4 sh_dec[kShare ? 2 : 1][kShare ? L : 1];
    __shared__ float sh_tok[kShare ? 2 : 1][4];
    auto widen = [&](const TokenIn &in, Token &w, int t) {
        if constexpr (kShare) {
            const int par = t & 1;
            w.q[0] = in.q[0].get();
            w.k[0] = in.k[0].get();
            const float4 gv = in.g[0].get();
            if (wave < kNormWave) {
                // this row group's channel 4 kc + r, r = rgw < 4
                const int r = rgw;
                const float x = r == 0 ? gv.x : r == 1 ? gv.y : r == 2 ? gv.z : gv.w;
                float d;
                if constexpr (GATE == KDA_GATE_RAW) {
                    const float db = r == 0 ? dtb[0].x : r == 1 ? dtb[0].y : r == 2 ? dtb[0].z : dtb[0].w;
                    d = expf(a.lower_bound / (1.0f + expf(-(expA * (x + db)))));
                } else {
                    d = expf(x);
                }
                reinterpret_cast<float *>(&sh_dec[par][kc])[r] = d;
            } else if (wave == kNormWave) {
                if (norm) {
                    const bool kr_group = (rgw & 1) != 0;
                    float s = 0.f;
                    s += kr_group ? dot4(w.k[0], w.k[0]) : dot4(w.q[0], w.q[0]);
                    s = group_sum<L>(s);
                    const float inv = 1.0f / sqrtf(s + 1e-6f);
                    if (kc == 0 && rgw < 4 + 2) {
                        sh_tok[par][kr_group ? 1 : 0] = kr_group ? inv : inv * a.scale;
                    }
                }
            } else if (wave == kNormWave + 1) {
                if (kc == 0 && (rgw & (RPW - 1)) == 0) {
                    if constexpr (GATE == KDA_GATE_RAW) {
                        sh_tok[par][2] = 1.0f / (1.0f + expf(-in.b));
                    } else {
                        sh_tok[par][2] = in.b;
                    }
                }
            }
            __syncthreads();
            w.dec[0] = sh_dec[par][kc];
            w.beta = sh_tok[par][2];
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                w.v[p] = in.v.get(p);
            }
            float qsc = a.scale;
            if (norm) {
                qsc = sh_tok[par][0];
                const float kr = sh_tok[par][1];
                w.k[0] = make_float4(w.k[0].x * kr, w.k[0].y * kr, w.k[0].z * kr, w.k[0].w * kr);
            }
            w.q[0] = make_float4(w.q[0].x * qsc, w.q[0].y * qsc, w.q[0].z * qsc, w.q[0].w * qsc);
            return;
        }
#pragma unroll
        for (int j = 0; j < EV; ++j) {
            w.q[j] = in.q[j].get();
            w.k[j] = in.k[j].get();
            const float4 gv = in.g[j].get();
            if constexpr (GATE == KDA_GATE_RAW) {
                // g = lower_bound / (1 + exp(-(exp(A_log) * (a + dt_bias)))), decay = exp(g)
                const float lb = a.lower_bound;
                w.dec[j].x = expf(lb / (1.0f + expf(-(expA * (gv.x + dtb[j].x)))));
                w.dec[j].y = expf(lb / (1.0f + expf(-(expA * (gv.y + dtb[j].y)))));
                w.dec[j].z = expf(lb / (1.0f + expf(-(expA * (gv.z + dtb[j].z)))));
                w.dec[j].w = expf(lb / (1.0f + expf(-(expA * (gv.w + dtb[j].w)))));
            } else if constexpr (GATE == KDA_GATE_LOG) {
                w.dec[j] = make_float4(expf(gv.x), expf(gv.y), expf(gv.z), expf(gv.w));
            } else {
                w.dec[j] = gv;
            }
        }
        if constexpr (GATE == KDA_GATE_RAW) {
            w.beta = 1.0f / (1.0f + expf(-in.b));
        } else {
            w.beta = in.b;
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            w.v[p] = in.v.get(p);
        }
        float qsc = a.scale;
        if (norm) {
            // x / sqrt(sum x^2 + 1e-6), eps inside the sqrt; q then scaled.
            float qs = 0.f, ks = 0.f;
#pragma unroll
            for (int j = 0; j < EV; ++j) {
                qs += dot4(w.q[j], w.q[j]);
                ks += dot4(w.k[j], w.k[j]);
            }
            qs = group_sum<L>(qs);
            ks = group_sum<L>(ks);
            const float kr = 1.0f / sqrtf(ks + 1e-6f);
            qsc = (1.0f / sqrtf(qs + 1e-6f)) * a.scale;
#pragma unroll
            for (int j = 0; j < EV; ++j) {
                w.k[j] = make_float4(w.k[j].x * kr, w.k[j].y * kr, w.k[j].z * kr, w.k[j].w * kr);
            }
        }
#pragma unroll
        for (int j = 0; j < EV; ++j) {
            w.q[j] = make_float4(w.q[j].x * qsc, w.q[j].y * qsc, w.q[j].z * qsc, w.q[j].w * qsc);
        }
    };
    // sum over the lane's E elements of s * x, one multiply-add chain
    auto dot_lane = [](const float4 (&sv)[EV], const float4 (&xv)[EV]) {
        float acc = dot4(sv[0], xv[0]);
#pragma unroll
        for (int j = 1; j < EV; ++j) {
            acc = fmaf(sv[j].x, xv[j].x, acc);
            acc = fmaf(sv[j].y, xv[j].y, acc);
            acc = fmaf(sv[j].z, xv[j].z, acc);
            acc = fmaf(sv[j].w, xv[j].w, acc);
        }
        return acc;
    };
    auto step = [&](const Token &w, int t) {
        float pred[NP];
#pragma unroll
        for (int p = 0; p < NP; ++p) {
#pragma unroll
            for (int j = 0; j < EV; ++j) {
                S[p][j].x *= w.dec[j].x;
                S[p][j].y *= w.dec[j].y;
                S[p][j].z *= w.dec[j].z;
                S[p][j].w *= w.dec[j].w;
            }
            pred[p] = dot_lane(S[p], w.k);
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            pred[p] = group_sum<L>(pred[p]);
        }
        float o[NP];
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const float d = (w.v[p] - pred[p]) * w.beta;
#pragma unroll
            for (int j = 0; j < EV; ++j) {
                S[p][j].x += w.k[j].x * d;
                S[p][j].y += w.k[j].y * d;
                S[p][j].z += w.k[j].z * d;
                S[p][j].w += w.k[j].w * d;
            }
            o[p] = dot_lane(S[p], w.q);
        }
        const int step_i = t - bos;
        if (save_mid && step_i < a.mid_steps) {
            store_state(a.intermediate + n * a.mid_stride_req + step_i * a.mid_stride_step +
                            static_cast<int64_t>(head) * a.mid_stride_head,
                        false);
        }
        if (track_slot > 0 && step_i + 1 == track_len) {
            store_state(a.state + track_slot * a.state_stride_slot + head_off, vpool);
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            o[p] = group_sum<L>(o[p]);
        }
        // every lane of the row group holds the sums
        store_row<TV, NP, RS>(op + (static_cast<int64_t>(t) * H + head) * D + row0, o, kc);
    };
    // Two buffers, the second loaded only when a next token exists (an
    // unconditional reload would double the token loads of a decode step).
    TokenIn cur, nxt;
    if (bos < eos) {
        fetch(bos, cur);
    }
    for (int t = bos; t < eos; ++t) {
        if (t + 1 < eos) {
            fetch(t + 1, nxt);
        }
        Token w;
        widen(cur, w, t);
        step(w, t);
        cur = nxt;
    }

    // Tokens no sequence covers are zero (the reference allocates
    // zeros_like(v), kda_varlen_recurrent.cpp:142): the first request zeroes
    // [0, cu[0]) and the last one [cu[N], T). The DECAY form writes a
    // caller-owned output and touches only the rows its requests cover, as
    // the reference's prepared kernels do (prepared_recurrent.cpp:386-560),
    // so a caller may launch request by request into one buffer.
    auto zero_rows = [&](int t0, int t1) {
        float z[NP];
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            z[p] = 0.f;
        }
        for (int t = t0; t < t1; ++t) {
            store_row<TV, NP, RS>(op + (static_cast<int64_t>(t) * H + head) * D + row0, z, kc);
        }
    };
    if constexpr (GATE != KDA_GATE_DECAY) {
        if (n == 0) {
            zero_rows(0, bos);
        }
        if (n == a.num_seqs - 1) {
            zero_rows(eos, T);
        }
    }

    if (a.intermediate == nullptr && slot > 0) {
        store_state(a.state + slot * a.state_stride_slot + head_off, vpool);
    }
}

// ---------------------------------------------------------------------------
// Several tokens per sequence (verify, short prefill): tokens in blocks.
//
// What bounds the token loop is VALU issue: four multiply-adds per state
// element and token (65 us for 1169 tokens on 32 heads at the unpacked fp32
// rate), and before them the token's gates and norms, which every row group
// of the workgroup needs alike (about 350 of 550 instructions per token and
// wave when each forms them for itself). So they are formed once per
// workgroup: of a block of 16 tokens, 16-lane row group i loads token i (q,
// k, gate, beta and the tile's v rows), forms the decays, the normalized k
// and the scaled q, and leaves them in LDS; after one barrier every row group
// steps through the block's tokens reading ready values. The next block's
// inputs are loaded behind the barrier and wait in registers while the tokens
// run, and a token's outputs replace its v values in LDS, from where the
// block's rows leave as vectors. 16 requests of 20-120 tokens, H=32, raw
// gates: 253 -> 115 us; 2 x 63 tokens, H=4, D=64, fp32: 42 -> 17 us; 256 x 8
// tokens, H=32: 307 -> 210 us.
//
// SW: the waves that share a block. 4: the workgroup, 16 tokens a block. 1:
// each wave for its own rows, four tokens a block and no barrier, for few
// tokens on many pairs, where the state's traffic is the bound and a barrier
// only makes the waves' loads wait for each other.
// Row groups of 16 lanes, a lane owning D / 16 K elements of NP consecutive
// rows; a workgroup covers 16 NP rows.
// ---------------------------------------------------------------------------

template <int D, int NP, int SW, typename TQK, typename TV, int GATE>
__global__ __launch_bounds__(kThreads) void recurrent_block_kernel(const RecurrentLaunch a) {
    constexpr int L = 16;
    constexpr int EV = D / L / 4;  // 16-byte vectors per lane and row
    constexpr int RB = 16 * NP;    // rows per workgroup
    constexpr int VT = D / RB;     // workgroups per (sequence, head)
    constexpr int BTOK = 4 * SW;   // tokens per block: a row group of the sharing waves each
    constexpr int SR = BTOK * NP;  // rows of the sharing waves
    constexpr int VP = SR / L;     // v values a lane stages
    static_assert(D % RB == 0 && (SW == 1 || SW == 4) && VP >= 1, "whole row tiles");
    // D = 64 keeps its one-token form's expf (about 1 ulp); at D = 128 the one-token
    // form uses expf too, so there a token's state and output depend in their last bits
    // on whether the batch holds more than one token per request.
    auto dexp = [](float x) { return D == 128 ? fexp(x) : expf(x); };

    // one block's prepared tokens: [token][channel], and [token][row of the
    // tile]: v before the token's step, its output after
    __shared__ float4 all_k[4 / SW][BTOK][D / 4];
    __shared__ float4 all_q[4 / SW][BTOK][D / 4];
    __shared__ float4 all_dec[4 / SW][BTOK][D / 4];
    __shared__ float all_beta[4 / SW][BTOK];
    __shared__ alignas(16) float all_vo[4 / SW][BTOK][SR];

    const int H = a.num_heads;
    const int HC = a.head_count;
    // XCD-aware order, as in recurrent_kernel
    const int b = blockIdx.x;
    const int rest = b >> 3;
    const int vt = VT == 1 ? 0 : rest % VT;
    const int pair = VT == 1 ? b : (rest / VT) * 8 + (b & 7);
    const int n = pair / HC;
    const int head = a.head_begin + (pair - n * HC);
    if (n >= a.num_seqs) {
        return;
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kc = lane % L;
    // row group among the sharing waves; in the prologue, the block's token
    const int rg = SW == 1 ? lane / L : static_cast<int>(threadIdx.x) / L;
    const int share = SW == 1 ? wave : 0;
    const int base0 = vt * RB + share * SR;  // the sharing waves' first row
    const int row0 = base0 + rg * NP;
    auto &sh_k = all_k[share];
    auto &sh_q = all_q[share];
    auto &sh_dec = all_dec[share];
    auto &sh_beta = all_beta[share];
    auto &sh_vo = all_vo[share];
    auto sync = [&]() {
        if constexpr (SW == 4) {
            lds_barrier();
        } else {
            // one wave's LDS accesses happen in order
            asm volatile("" ::: "memory");
        }
    };
    const int T = a.num_tokens;

    const int2 ends = a.cu_pair(n);
    int slot = a.slot_index(n);
    int bos = ends.x;
    int eos = ends.y;
    bos = bos < 0 ? 0 : (bos > T ? T : bos);
    eos = eos < bos ? bos : (eos > T ? T : eos);
    if (slot < 0 || static_cast<int64_t>(slot) >= a.num_slots) {
        slot = 0;
    }

    auto koff = [&](int j) { return 4 * kc + 4 * L * j; };
    const TQK *qp = static_cast<const TQK *>(a.q);
    const TQK *kp = static_cast<const TQK *>(a.k);
    const TV *vp = static_cast<const TV *>(a.v);
    TV *op = static_cast<TV *>(a.out);
    using TG = typename std::conditional<GATE == KDA_GATE_RAW, uint16_t, float>::type;
    const TG *gp = static_cast<const TG *>(a.gate);

    // Inputs of this row group's token of the block at t0 (the last token's
    // where the block has fewer: loaded, prepared and never used). A wave
    // none of whose four tokens exists loads nothing.
    Raw4<TQK> rq[EV], rk[EV];
    Raw4<TG> rgate[EV];
    RowIn<TV, VP, VP == 1 ? 16 : 1> rv;
    // v and out may sit anywhere: whole vectors where both are aligned for
    // them, element by element otherwise
    constexpr uintptr_t kVecBytes = VP * sizeof(TV) > 16 ? 16 : VP * sizeof(TV);
    const bool vec = ((reinterpret_cast<uintptr_t>(vp) | reinterpret_cast<uintptr_t>(op)) & (kVecBytes - 1)) == 0;
    float rb = 0.f;
    auto fetch = [&](int t0) {
        if (t0 + (SW == 1 ? 0 : 4 * wave) < eos) {
            const int t = t0 + rg < eos ? t0 + rg : eos - 1;
            const int64_t bi = static_cast<int64_t>(t) * H + head;
            const int64_t base = bi * D;
#pragma unroll
            for (int j = 0; j < EV; ++j) {
                rq[j].load(qp + base + koff(j));
                rk[j].load(kp + base + koff(j));
                rgate[j].load(gp + base + koff(j));
            }
            if (vec) {
                rv.load(vp + base + base0 + kc * VP);
            } else {
                rv.load_each(vp + base + base0 + kc * VP);
            }
            if constexpr (GATE == KDA_GATE_RAW) {
                rb = bf16_to_f32(static_cast<const uint16_t *>(a.beta)[bi]);
            } else {
                rb = static_cast<const float *>(a.beta)[bi];
            }
        }
    };
    // Raw gates: the inputs' loads go ahead of the state's, whose wait would
    // otherwise cover them, since the prologue is long (512 x 2 tokens, H=32,
    // one wave sharing: 356 us, against 377 behind them). Prepared gates have
    // a short prologue, and with one wave sharing the state goes first
    // (1024 x 4 tokens, H=16: 373 us, against 389).
    constexpr bool kInputsFirst = SW == 4 || GATE == KDA_GATE_RAW;
    if (kInputsFirst && bos < eos) {
        fetch(bos);
    }

    const int64_t head_off = static_cast<int64_t>(head) * a.state_stride_head;
    const bool vpool = GATE == KDA_GATE_DECAY && a.state_v_contiguous != 0;
    float4 S[NP][EV];
    if (slot > 0) {
        const float *src = a.state + slot * a.state_stride_slot + head_off;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
#pragma unroll
            for (int j = 0; j < EV; ++j) {
                if (vpool) {
                    const float *e = src + static_cast<int64_t>(koff(j)) * D + row0 + p;
                    S[p][j] = make_float4(e[0], e[D], e[2 * D], e[3 * D]);
                } else {
                    S[p][j] = load4_stream(src + static_cast<int64_t>(row0 + p) * D + koff(j));
                }
            }
        }
    } else {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
#pragma unroll
            for (int j = 0; j < EV; ++j) {
                S[p][j] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
    }

    if (!kInputsFirst && bos < eos) {
        fetch(bos);
    }

    int track_slot = 0;
    int track_len = -1;
    if (a.track_indices != nullptr) {
        track_slot = a.track_index(n);
        if (track_slot <= 0 || static_cast<int64_t>(track_slot) >= a.num_slots) {
            track_slot = 0;
        } else {
            track_len = a.track_length(n);
        }
    }
    // The stores' addresses are formed where they are used: hoisted out of the token
    // loop (three places store a state, in two layouts with decay gates) they cost 20
    // to 40 registers, and with fp32 inputs a workgroup per CU: 64-row tiles took 138
    // to 144, three per CU (512 x 3 tokens, decay gates: 17.3 us; now up to 120 and
    // four: 14.2), 128-row ones 170 to 176, two. The others have room for them, and at
    // many pairs fewer waves stream the states better (8192 x 2, 32-row tiles: 177
    // us with four workgroups per CU, 184 with five).
    constexpr bool kFormHere = GATE == KDA_GATE_DECAY || (sizeof(TQK) == 4 && NP >= 4);
    auto store_state = [&](float *dst, bool vlayout) {
        int rs = row0;
        int ks = 4 * kc;
        if constexpr (kFormHere) {
            asm volatile("" : "+v"(rs), "+v"(ks));
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) {
#pragma unroll
            for (int j = 0; j < EV; ++j) {
                if (vlayout) {
                    float *e = dst + static_cast<int64_t>((ks + 4 * L * j)) * D + rs + p;
                    e[0] = S[p][j].x;
                    e[D] = S[p][j].y;
                    e[2 * D] = S[p][j].z;
                    e[3 * D] = S[p][j].w;
                } else {
                    store4_stream(dst + static_cast<int64_t>(rs + p) * D + (ks + 4 * L * j), S[p][j]);
                }
            }
        }
    };
    if (track_slot > 0 && track_len == 0) {
        store_state(a.state + track_slot * a.state_stride_slot + head_off, vpool);
    }

    float expA = 0.f;
    if constexpr (GATE == KDA_GATE_RAW) {
        expA = expf(a.A_log[head]);
    }
    const bool norm = (GATE == KDA_GATE_RAW) || (a.qk_l2norm != 0);
    const bool save_mid = a.intermediate != nullptr && slot > 0 && n < a.mid_rows;

    // the fetched token, prepared, into LDS
    auto prepare = [&](int t0) {
        if (t0 + (SW == 1 ? 0 : 4 * wave) >= eos) {
            return;
        }
        float4 q[EV], k[EV], dec[EV];
#pragma unroll
        for (int j = 0; j < EV; ++j) {
            q[j] = rq[j].get();
            k[j] = rk[j].get();
            const float4 gv = rgate[j].get();
            if constexpr (GATE == KDA_GATE_RAW) {
                // g = lower_bound / (1 + exp(-(exp(A_log) * (a + dt_bias)))), decay = exp(g)
                const float lb = a.lower_bound;
                const float4 dtb = load4(a.dt_bias + static_cast<int64_t>(head) * D + koff(j));
                dec[j].x = dexp(lb / (1.0f + dexp(-(expA * (gv.x + dtb.x)))));
                dec[j].y = dexp(lb / (1.0f + dexp(-(expA * (gv.y + dtb.y)))));
                dec[j].z = dexp(lb / (1.0f + dexp(-(expA * (gv.z + dtb.z)))));
                dec[j].w = dexp(lb / (1.0f + dexp(-(expA * (gv.w + dtb.w)))));
            } else if constexpr (GATE == KDA_GATE_LOG) {
                dec[j] = make_float4(dexp(gv.x), dexp(gv.y), dexp(gv.z), dexp(gv.w));
            } else {
                dec[j] = gv;
            }
        }
        float qsc = a.scale;
        float kr = 1.f;
        if (norm) {
            // x / sqrt(sum x^2 + 1e-6), eps inside the sqrt; q then scaled.
            float qs = 0.f, ks = 0.f;
#pragma unroll
            for (int j = 0; j < EV; ++j) {
                qs += dot4(q[j], q[j]);
                ks += dot4(k[j], k[j]);
            }
            qs = group_sum<L>(qs);
            ks = group_sum<L>(ks);
            kr = 1.0f / sqrtf(ks + 1e-6f);
            qsc = (1.0f / sqrtf(qs + 1e-6f)) * a.scale;
        }
#pragma unroll
        for (int j = 0; j < EV; ++j) {
            sh_k[rg][kc + L * j] = make_float4(k[j].x * kr, k[j].y * kr, k[j].z * kr, k[j].w * kr);
            sh_q[rg][kc + L * j] = make_float4(q[j].x * qsc, q[j].y * qsc, q[j].z * qsc, q[j].w * qsc);
            sh_dec[rg][kc + L * j] = dec[j];
        }
#pragma unroll
        for (int p = 0; p < VP; ++p) {
            sh_vo[rg][kc * VP + p] = rv.get(p);
        }
        if (kc == 0) {
            if constexpr (GATE == KDA_GATE_RAW) {
                sh_beta[rg] = 1.0f / (1.0f + dexp(-rb));
            } else {
                sh_beta[rg] = rb;
            }
        }
    };
    struct Token {
        float4 k[EV], dec[EV], q[EV];
        float beta;
        float v[NP];
    };
    auto read = [&](Token &w, int i) {
#pragma unroll
        for (int j = 0; j < EV; ++j) {
            w.dec[j] = sh_dec[i][kc + L * j];
            w.k[j] = sh_k[i][kc + L * j];
            w.q[j] = sh_q[i][kc + L * j];
        }
        w.beta = sh_beta[i];
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            w.v[p] = sh_vo[i][rg * NP + p];
        }
    };
    // sum over the lane's elements of s * x, one multiply-add chain
    auto dot_lane = [](const float4 (&sv)[EV], const float4 (&xv)[EV]) {
        float acc = dot4(sv[0], xv[0]);
#pragma unroll
        for (int j = 1; j < EV; ++j) {
            acc = fmaf(sv[j].x, xv[j].x, acc);
            acc = fmaf(sv[j].y, xv[j].y, acc);
            acc = fmaf(sv[j].z, xv[j].z, acc);
            acc = fmaf(sv[j].w, xv[j].w, acc);
        }
        return acc;
    };
    auto step = [&](const Token &w, int i, int step_i) {
        float pred[NP];
#pragma unroll
        for (int p = 0; p < NP; ++p) {
#pragma unroll
            for (int j = 0; j < EV; ++j) {
                S[p][j].x *= w.dec[j].x;
                S[p][j].y *= w.dec[j].y;
                S[p][j].z *= w.dec[j].z;
                S[p][j].w *= w.dec[j].w;
            }
            pred[p] = dot_lane(S[p], w.k);
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            pred[p] = group_sum<L>(pred[p]);
        }
        float o[NP];
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const float d = (w.v[p] - pred[p]) * w.beta;
#pragma unroll
            for (int j = 0; j < EV; ++j) {
                S[p][j].x += w.k[j].x * d;
                S[p][j].y += w.k[j].y * d;
                S[p][j].z += w.k[j].z * d;
                S[p][j].w += w.k[j].w * d;
            }
            o[p] = dot_lane(S[p], w.q);
        }
        if (save_mid && step_i < a.mid_steps) {
            store_state(a.intermediate + n * a.mid_stride_req + step_i * a.mid_stride_step +
                            static_cast<int64_t>(head) * a.mid_stride_head,
                        false);
        }
        if (track_slot > 0 && step_i + 1 == track_len) {
            store_state(a.state + track_slot * a.state_stride_slot + head_off, vpool);
        }
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            o[p] = group_sum<L>(o[p]);
        }
        if (kc == 0) {  // every lane of the row group holds the sums
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                sh_vo[i][rg * NP + p] = o[p];
            }
        }
    };
    // the final state, ahead of the last block's outputs
    auto finish = [&]() {
        if (a.intermediate == nullptr && slot > 0) {
            store_state(a.state + slot * a.state_stride_slot + head_off, vpool);
        }
    };
    if (bos >= eos) {
        finish();
    }
    for (int t0 = bos; t0 < eos; t0 += BTOK) {
        prepare(t0);
        sync();
        if (t0 + BTOK < eos) {
            fetch(t0 + BTOK);
        }
        const int len = eos - t0 < BTOK ? eos - t0 : BTOK;
        if constexpr (NP == 1) {
            Token cur;
            read(cur, 0);
            for (int i = 0; i < len; ++i) {
                Token nxt;
                read(nxt, i + 1 < len ? i + 1 : i);
                step(cur, i, t0 - bos + i);
                cur = nxt;
            }
        } else {
            for (int i = 0; i < len; ++i) {
                Token cur;
                read(cur, i);
                step(cur, i, t0 - bos + i);
            }
        }
        if (t0 + BTOK >= eos) {
            finish();
        }
        sync();
        // the block's outputs, token rg by row group rg, which also rewrites
        // exactly these entries for the next block
        if (rg < len) {
            float o[VP];
#pragma unroll
            for (int p = 0; p < VP; ++p) {
                o[p] = sh_vo[rg][kc * VP + p];
            }
            TV *dst = op + (static_cast<int64_t>(t0 + rg) * H + head) * D + base0 + kc * VP;
            if (VP > 1 && vec) {
                store_row<TV, VP, VP == 1 ? 16 : 1>(dst, o, kc);
            } else {
#pragma unroll
                for (int p = 0; p < VP; ++p) {
                    store1(dst + p, o[p]);
                }
            }
        }
    }

    // rows no request covers, as in recurrent_kernel
    auto zero_rows = [&](int ta, int tb) {
        for (int t = ta + rg; t < tb; t += BTOK) {
#pragma unroll
            for (int p = 0; p < VP; ++p) {
                store1(op + (static_cast<int64_t>(t) * H + head) * D + base0 + kc * VP + p, 0.f);
            }
        }
    };
    if constexpr (GATE != KDA_GATE_DECAY) {
        if (n == 0) {
            zero_rows(0, bos);
        }
        if (n == a.num_seqs - 1) {
            zero_rows(eos, T);
        }
    }

}

using KernelFn = void (*)(const RecurrentLaunch);

// Tile shapes, by the rows a workgroup covers.
enum Shape {
    kDecode16, kDecode8, kBlock16, kBlock32, kBlock64, kBlock128, kWave64, kWave128, kD64Small, kD64Large
};

template <int D, typename TQK, typename TV, int GATE>
KernelFn pick_shape(Shape shape) {
    if constexpr (D == 128) {
        switch (shape) {
            case kDecode16: return recurrent_kernel<D, 32, 2, TQK, TV, GATE>;
            case kDecode8: return recurrent_kernel<D, 32, 1, TQK, TV, GATE>;
            case kBlock16: return recurrent_block_kernel<D, 1, 4, TQK, TV, GATE>;
            case kBlock32: return recurrent_block_kernel<D, 2, 4, TQK, TV, GATE>;
            case kBlock64: return recurrent_block_kernel<D, 4, 4, TQK, TV, GATE>;
            case kBlock128: return recurrent_block_kernel<D, 8, 4, TQK, TV, GATE>;
            default: break;
        }
        if constexpr (GATE == KDA_GATE_RAW) {  // prepared gates are not launched with these
            switch (shape) {
                case kWave64: return recurrent_block_kernel<D, 4, 1, TQK, TV, GATE>;
                case kWave128: return recurrent_block_kernel<D, 8, 1, TQK, TV, GATE>;
                default: break;
            }
        }
        return nullptr;
    } else {
        switch (shape) {
            case kD64Large: return recurrent_kernel<D, 16, 4, TQK, TV, GATE>;
            case kD64Small: return recurrent_kernel<D, 16, 1, TQK, TV, GATE>;
            case kBlock16: return recurrent_block_kernel<D, 1, 4, TQK, TV, GATE>;
            case kBlock64: return recurrent_block_kernel<D, 4, 4, TQK, TV, GATE>;
            default: return nullptr;
        }
    }
}

template <int D>
KernelFn pick_kernel(int gate, int qk_dtype, int v_dtype, Shape shape) {
    if (gate == KDA_GATE_RAW) {
        if (qk_dtype == KDA_BF16 && v_dtype == KDA_BF16) {
            return pick_shape<D, uint16_t, uint16_t, KDA_GATE_RAW>(shape);
        }
        return nullptr;
    }
    if (gate == KDA_GATE_LOG) {
        if (qk_dtype == KDA_BF16 && v_dtype == KDA_BF16) {
            return pick_shape<D, uint16_t, uint16_t, KDA_GATE_LOG>(shape);
        }
        if (qk_dtype == KDA_F32 && v_dtype == KDA_F32) {
            return pick_shape<D, float, float, KDA_GATE_LOG>(shape);
        }
        return nullptr;
    }
    if (gate == KDA_GATE_DECAY) {
        if (qk_dtype == KDA_F32 && v_dtype == KDA_BF16) {
            return pick_shape<D, float, uint16_t, KDA_GATE_DECAY>(shape);
        }
        if (qk_dtype == KDA_F32 && v_dtype == KDA_F32) {
            return pick_shape<D, float, float, KDA_GATE_DECAY>(shape);
        }
        return nullptr;
    }
    return nullptr;
}

// The tile shape, by tokens per sequence (their mean) and (sequence, head) pairs.
// Measured on MI355X as graph replays over pools that rotate through 1 GiB, in
// microseconds, raw gates on bf16, log gates on bf16 and fp32 and decay gates at
// 64 to 16384 pairs and 2 to 16 tokens (ragged: 20 to 120); "loop" is a token loop
// without shared blocks, which the block shapes replaced.
//
// One token (decode), D = 128: 32-lane rows, 2 rows per lane: 16-row tiles, eight
// workgroups per pair, which stream the state fastest (256 x 1, H=32: 173,
// against 182 with 32-row tiles; 96 x 1, log gates: 4.4, against 5.6 with 8-row
// tiles, raw 5.1 against 5.9); 8-row tiles below 48 pairs (16: 3.1 against 3.2; 48:
// 3.9 against 3.8) and, on a pool of V-contiguous rows, below 128 (72: 8.7
// against 9.0).
//
// Several tokens, D = 128. What a tile shares is the token's preparation: long with
// raw gates (four exponentials and a reciprocal per channel, the norms), short with
// prepared ones. Below that, what counts is how many workgroups there are, whether
// all are resident at once (256 CUs hold 256 pairs of 32-row tiles, 512 of 64-row
// ones, 768 of 128-row ones), and how they stream the states.
Shape tile_shape(const KdaRecurrentArgs &a, int64_t pairs) {
    const int64_t seqs = a.num_seqs;
    const int64_t ntok = a.num_tokens;
    auto tokens = [&](int n) { return ntok <= n * seqs; };  // up to n a sequence
    if (a.head_dim != 128) {
        // 64-row tiles are one workgroup per pair, 16-row tiles four (2 x 37-63
        // tokens, H=4: 17 against 25; 64 x 4, H=16: 14.9 against 9.1)
        if (tokens(1)) {
            return pairs >= 2048 ? kD64Large : kD64Small;
        }
        return pairs >= 256 ? kBlock64 : kBlock16;
    }
    // a pool of V-contiguous rows moves in 4-byte pieces
    const bool vpool = a.gate_mode == KDA_GATE_DECAY && a.state_v_contiguous != 0;
    if (tokens(1)) {
        return pairs < (vpool ? 128 : 48) ? kDecode8 : kDecode16;
    }
    if (a.gate_mode == KDA_GATE_RAW) {
        // few pairs: 16-row tiles spread a step over most CUs (32 x 4: 5.13, 32-row
        // tiles 5.15, loop 6.1), from 48 pairs 32-row tiles fill them with half the
        // preparations (48 x 2: 4.8 against 5.2; 256 x 2: 8.0 against 8.8 with
        // 64-row tiles, loop 8.5; 256 x 20-120: 63 against 82, loop 170). Up to 64 pairs
        // 32-row tiles are at most one workgroup per CU, and nothing then shares a CU
        // with the longest sequence: past verify lengths, prompts of unlike lengths take
        // 16-row tiles (36 x 20-120: 39-45 against 42-49, 64 x 4-40: 12.6-19.7 against
        // 13.8-19.5), and prompts of one length pay for it (64 x 100: 44.8 against 42.6)
        if (pairs <= 32 || (pairs <= 64 && !tokens(8))) {
            return kBlock16;
        }
        if (pairs <= 256) {
            return kBlock32;
        }
        // 512 x 2: 13.9, 128-row tiles 14.5, loop 17.1; 512 x 16: 29.2, 30.9,
        // loop 57; long sequences, bound by VALU issue, stay with their
        // occupancy (2048 x 20-120: 401 against 418, loop 728)
        if (pairs <= 512 || !tokens(16)) {
            return kBlock64;
        }
        // 128-row tiles prepare a token once per pair (640 x 2: 16.1 against 19.8
        // with 64-row tiles, loop 19.3; 1536 x 4: 42.2, 45.1, 46.3; 4096 x 6:
        // 108.6, 109.0, 131). From 2048 pairs the state's traffic bounds up to
        // four tokens, and a barrier only couples the waves' loads (one wave
        // sharing, 4096 x 2: 95.9 against 104, loop 96.6; 4096 x 4: 99.4, 105.5,
        // 107). At two tokens the third round of 128-row tiles is short just
        // below that (1856 x 2: 48.6 with one wave sharing 64-row tiles, against
        // 49.9, loop 47.8).
        if (tokens(2) && pairs >= 1792 && pairs < 2048) {
            return kWave64;
        }
        return pairs < 2048 || !tokens(4) ? kBlock128 : kWave128;
    }
    // Prepared gates: 16-row tiles up to 128 pairs (128 x 2: 4.8, 32-row tiles 5.1,
    // loop 5.9), 32-row tiles up to 256 (256 x 4: 8.4, 64-row tiles 8.6, loop 9.2;
    // 256 x 16: 14.9, 16.9, loop 19.6)
    if (pairs <= 128) {
        return kBlock16;
    }
    const bool decay = a.gate_mode == KDA_GATE_DECAY;
    // V-contiguous rows: a tile of 32 takes whole lines, taller ones touch them
    // once per row (1024 x 2: 72 with 32-row tiles, 73 with 64-row, 131 with 128-row
    // tiles, loop 79; 2048 x 8: 141, 149, 250, 261)
    // (decay gates' are five per CU: 320 x 4: 9.9, 64-row tiles 11.0, loop 12.0)
    if (pairs <= (decay ? 320 : 256) || (vpool && tokens(8))) {
        return kBlock32;
    }
    if (vpool) {
        return kBlock64;
    }
    // 384 x 4: 64-row tiles 10.2, 32-row tiles 13.1, 128-row tiles 12.0, loop 11.9
    // (decay gates 11.9, 14.8, 14.3, 13.0)
    if (pairs <= 384) {
        return kBlock64;
    }
    // 512 x 2: log gates 12.6 with 128-row tiles, 64-row tiles 15.0, loop 17.0; 512 x
    // 8: 18.8, 16.4, 20.3; decay gates, 2: 16.9, 13.7, 17.8; 8: 22.3, 19.0, 21.1
    if (pairs <= 512) {
        return !decay && tokens(4) ? kBlock128 : kBlock64;
    }
    // 640 x 4: log gates 15.6 with 128-row tiles, 32-row tiles 18.6, loop 21.2;
    // fp32 16.1, 20.2, 21.3; decay gates 20.4, 21.1, 23.7
    if (pairs <= 768 && tokens(decay ? 4 : 6)) {
        return kBlock128;
    }
    // Many pairs: 32-row tiles stream a few tokens' states best (2048 x 4: 48.3,
    // 64-row tiles 50.8, 128-row tiles 52.8, loop 53.1; decay gates 55.6, 57.2, 60.4,
    // 61.6; 8192 x 2: 177, 199, 191, 184); more tokens take the 64-row ones (16384 x
    // 6: 396, 406; decay gates, 2048 x 16: 94, 99) and log gates past eight
    // the 128-row ones (4096 x 16: 165, 64-row tiles 173, 32-row tiles 182)
    if (tokens(5)) {
        return kBlock32;
    }
    return !decay && !tokens(8) && tokens(16) ? kBlock128 : kBlock64;
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
bool aligned8(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; }

}  // namespace
}  // namespace kda

extern "C" int kda_recurrent_launch(const KdaRecurrentArgs *args, void *stream) {
    return kda_recurrent_launch_wide(args, 0, stream);
}

extern "C" int kda_recurrent_launch_wide(const KdaRecurrentArgs *args, int32_t wide, void *stream) {
    using namespace kda;
    if (args == nullptr || (wide & ~kWideAll) != 0) {
        return KDA_ERR_INVALID_ARGUMENT;
    }
    const KdaRecurrentArgs &a = *args;
    const int D = a.head_dim;
    if (D != 64 && D != 128) {
        return KDA_ERR_UNSUPPORTED;
    }
    if (a.state_v_contiguous != 0 && a.gate_mode != KDA_GATE_DECAY) {
        return KDA_ERR_UNSUPPORTED;  // the [K,V] pool is the prepared (DECAY) layout
    }
    if (a.num_seqs < 0 || a.num_tokens < 0 || a.num_heads <= 0 || a.num_slots < 0) {
        return KDA_ERR_INVALID_ARGUMENT;
    }
    if (a.num_seqs == 0) {
        return KDA_OK;
    }
    // token tensors are never read or written when there are no tokens
    const bool tokens = a.num_tokens > 0;
    if ((tokens && (a.q == nullptr || a.k == nullptr || a.v == nullptr || a.gate == nullptr ||
                    a.beta == nullptr || a.out == nullptr)) ||
        a.state == nullptr || a.state_indices == nullptr || a.cu_seqlens == nullptr) {
        return KDA_ERR_INVALID_ARGUMENT;
    }
    if (a.gate_mode == KDA_GATE_RAW && (a.A_log == nullptr || a.dt_bias == nullptr)) {
        return KDA_ERR_INVALID_ARGUMENT;
    }
    if ((a.track_indices == nullptr) != (a.track_lens == nullptr)) {
        return KDA_ERR_INVALID_ARGUMENT;
    }
    // 16-byte state vectors: pool base and strides must keep rows aligned.
    if (!aligned16(a.state) || (a.state_stride_slot & 3) || (a.state_stride_head & 3)) {
        return KDA_ERR_INVALID_ARGUMENT;
    }
    if (a.intermediate != nullptr &&
        (!aligned16(a.intermediate) || (a.mid_stride_req & 3) || (a.mid_stride_step & 3) ||
         (a.mid_stride_head & 3))) {
        return KDA_ERR_INVALID_ARGUMENT;
    }
    const bool qk_f32 = a.qk_dtype == KDA_F32;
    if (qk_f32 ? !(aligned16(a.q) && aligned16(a.k)) : !(aligned8(a.q) && aligned8(a.k))) {
        return KDA_ERR_INVALID_ARGUMENT;
    }
    if (a.gate_mode == KDA_GATE_RAW ? !aligned8(a.gate) : !aligned16(a.gate)) {
        return KDA_ERR_INVALID_ARGUMENT;
    }

    RecurrentLaunch kargs{{wide}, a};
    if (kargs.head_begin < 0 || kargs.head_begin >= kargs.num_heads || kargs.head_count < 0) {
        return KDA_ERR_INVALID_ARGUMENT;
    }
    if (kargs.head_count == 0 || kargs.head_begin + kargs.head_count > kargs.num_heads) {
        kargs.head_count = kargs.num_heads - kargs.head_begin;
    }
    const int64_t pairs = static_cast<int64_t>(a.num_seqs) * kargs.head_count;
    const Shape shape = tile_shape(a, pairs);
    int rows_per_wg = 128;
    switch (shape) {
        case kDecode8: rows_per_wg = 8; break;
        case kDecode16: case kBlock16: case kD64Small: rows_per_wg = 16; break;
        case kBlock32: rows_per_wg = 32; break;
        case kBlock64: case kWave64: case kD64Large: rows_per_wg = 64; break;
        case kBlock128: case kWave128: break;
    }
    KernelFn fn = (D == 128) ? pick_kernel<128>(a.gate_mode, a.qk_dtype, a.v_dtype, shape)
                             : pick_kernel<64>(a.gate_mode, a.qk_dtype, a.v_dtype, shape);
    if (fn == nullptr) {
        return KDA_ERR_UNSUPPORTED;
    }
    const int vts = D / rows_per_wg;
    const int64_t blocks = vts == 1 ? pairs : (pairs + 7) / 8 * 8 * vts;
    if (blocks > 0x7fffffff) {
        return KDA_ERR_INVALID_ARGUMENT;
    }
    void *params[] = {&kargs};
    const hipError_t err =
        hipLaunchKernel(reinterpret_cast<const void *>(fn), dim3(static_cast<unsigned>(blocks)),
                        dim3(kThreads), params, 0, static_cast<hipStream_t>(stream));
    return err == hipSuccess ? KDA_OK : KDA_ERR_LAUNCH;
}
