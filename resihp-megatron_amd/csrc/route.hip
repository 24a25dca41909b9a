// Routing kernels for gfx950: router logits + top-k + gates, the dispatch plan
// (histogram, scan, stable scatter), the expert-bias update and the router
// backward to the selected logits.
//
// Reference: resihp/runtime/moe.py:64-66 (bias update), :75-79 (route),
// :94 and :192 (bincount), :97 and :193-207 (dispatch order).
//
// Floating-point contraction is off in this file: every add and multiply is
// one IEEE operation, and the fused multiply-adds are written explicitly, so
// the logits, selection and gates are reproducible bit for bit.
#pragma clang fp contract(off)

#include <algorithm>
#include <mutex>
#include <string>
#include <type_traits>

#include "dma.h"

namespace rhp {
namespace {

constexpr int kThreads = 256;
constexpr int kEpt = 8;     // experts per thread in the logit phase
constexpr int kTpt = 4;     // tokens per thread in the logit phase
constexpr int kMaxE = 1024;

__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }

template <class AT> __device__ __forceinline__ AT neg_inf();
template <> __device__ __forceinline__ float neg_inf<float>() { return -__builtin_inff(); }
template <> __device__ __forceinline__ double neg_inf<double>() { return -__builtin_inf(); }

// Loads 8 consecutive elements of a row as the accumulation type.
template <class XT, class AT> struct Load8;
template <> struct Load8<bf16, float> {
    __device__ __forceinline__ static void run(const bf16* p, float* v) {
        uint4 q = *reinterpret_cast<const uint4*>(p);
        uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[2 * i] = __uint_as_float(w[i] << 16);
            v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
        }
    }
};
template <> struct Load8<float, float> {
    __device__ __forceinline__ static void run(const float* p, float* v) {
        float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    }
};
template <> struct Load8<double, double> {
    __device__ __forceinline__ static void run(const double* p, double* v) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            double2 a = reinterpret_cast<const double2*>(p)[i];
            v[2 * i] = a.x;
            v[2 * i + 1] = a.y;
        }
    }
};

// Layout of one routing block: TB tokens; each work item is (token group of kTpt
// tokens, segment s, expert chunk of kEpt experts).
struct RouteShape {
    int seg, S, n_ec, units, ntg, tb;
};

// Descending key, ties to the lowest expert id.
template <class AT> __device__ __forceinline__ bool better(AT va, int ia, AT vb, int ib) {
    return va > vb || (va == vb && ia < ib);
}

// v of the lane a DPP control picks (every lane takes part).
template <int CTRL> __device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL> __device__ __forceinline__ double dpp(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// Largest v of each aligned group of lpt lanes (a power of two), no NaN among
// them, in every lane of the group: lane exchanges within 16 lanes are DPP
// (quad swaps, then mirrored halves, whose lanes already agree).
template <class AT> __device__ __forceinline__ AT group_max(AT v, int lpt) {
    auto take = [&](AT o) { v = o > v ? o : v; };
    if (lpt > 1) take(dpp<0xB1>(v));    // quad_perm 1 0 3 2
    if (lpt > 2) take(dpp<0x4E>(v));    // quad_perm 2 3 0 1
    if (lpt > 4) take(dpp<0x141>(v));   // row_half_mirror
    if (lpt > 8) take(dpp<0x140>(v));   // row_mirror
    if (lpt > 16) take(__shfl_xor(v, 16, 64));
    if (lpt > 32) take(__shfl_xor(v, 32, 64));
    return v;
}

// Selection and gates of a block's tb tokens (first token t_block) from their
// logits in LDS, token tl's at lg + tl ld; sel[tb][k] and num[tb][k] are LDS
// scratch.  nthreads: block size.
//   A group of lpt lanes selects a token's experts: the largest remaining key
// by lane exchange, its expert by a ballot (ties, rare, by a second pass over
// the ids).  Exchanging (key, id) pairs through LDS shuffles took 52 of 120 us
// at 16384 tokens, 64 experts, top 6.  A lane keeps the keys of its first two
// experts (all of them up to 128 experts) in registers.
//   Gates: one thread per (token, slot); sums in slot order.
template <class AT>
__device__ __forceinline__ void select_and_gate(const AT* lg, int ld, int* sel, AT* num, int64_t t_block, int tb,
                                                int nthreads, int64_t T, int E, int k, int score, int normalize,
                                                AT scale, const AT* __restrict__ bias, int32_t* __restrict__ topi,
                                                AT* __restrict__ gates) {
    const int tid = threadIdx.x;
    int lpt = 1;
    while (lpt < E && lpt < 64) lpt <<= 1;
    const int lane = tid & 63, wave = tid >> 6;
    const int gl = lane & (lpt - 1);
    const int groups_per_block = (nthreads / 64) * (64 / lpt);
    const int my_group = wave * (64 / lpt) + lane / lpt;
    const int cand = (E + lpt - 1) / lpt;   // each lane owns experts gl + c * lpt
    const int none = 0x7fffffff;
    const uint64_t group_lanes = (lpt == 64 ? ~0ull : (1ull << lpt) - 1) << (lane & ~(lpt - 1));
    for (int tl0 = 0; tl0 < tb; tl0 += groups_per_block) {
        const int tl = tl0 + my_group;
        const bool active = tl < tb && (t_block + tl) < T;
        auto key = [&](int c) {
            const int e = gl + c * lpt;
            if (!active || e >= E) return neg_inf<AT>();
            AT v = lg[tl * ld + e];
            if (score == RHP_SCORE_SIGMOID) v = rhp_sigmoid(v);
            if (bias) v = v + bias[e];
            return v != v ? neg_inf<AT>() : v;
        };
        const AT key0 = key(0), key1 = cand > 1 ? key(1) : neg_inf<AT>();
        uint32_t taken = 0;   // bit c: candidate c already chosen (cand <= 16 since E <= 1024)
        for (int j = 0; j < k; ++j) {
            AT bv = neg_inf<AT>();
            int bi = none;
            if (active) {
                for (int c = 0; c < cand; ++c) {
                    const int e = gl + c * lpt;
                    if (e >= E || ((taken >> c) & 1u)) continue;
                    const AT v = c == 0 ? key0 : c == 1 ? key1 : key(c);
                    if (better(v, e, bv, bi)) { bv = v; bi = e; }
                }
            }
            const AT m = group_max(bv, lpt);
            uint64_t win = __ballot(bi != none && bv == m) & group_lanes;
            int id = bi;
            if (__ballot(__popcll(win) > 1)) {   // a tie in some group of the wave: its lowest id
                int low = bi != none && bv == m ? bi : none;
                for (int o = lpt >> 1; o >= 1; o >>= 1) low = min(low, __shfl_xor(low, o, 64));
                id = low;
            }
            if (active && bi == id && ((win >> lane) & 1)) {
                taken |= 1u << (id / lpt);
                sel[tl * k + j] = id;
            }
        }
    }
    __syncthreads();

    // num: the slot's exp (softmax, over the selected logits) or sigmoid.
    const int n = static_cast<int>(min<int64_t>(tb, T - t_block)) * k;
    for (int i = tid; i < n; i += nthreads) {
        const int tl = i / k;
        const AT* l = lg + tl * ld;
        const int* s = sel + tl * k;
        const AT v = l[s[i - tl * k]];
        if (score == RHP_SCORE_SOFTMAX) {
            AT m = l[s[0]];
            for (int j = 1; j < k; ++j) m = (l[s[j]] > m) ? l[s[j]] : m;
            num[i] = rhp_exp_t(v - m);
        } else {
            num[i] = rhp_sigmoid(v);
        }
    }
    __syncthreads();
    for (int i = tid; i < n; i += nthreads) {
        const AT* g = num + i / k * k;
        AT sum = g[0];
        for (int j = 1; j < k; ++j) sum = sum + g[j];
        const AT v = num[i];
        topi[t_block * k + i] = sel[i];
        gates[t_block * k + i] = (score == RHP_SCORE_SOFTMAX || normalize ? v / sum : v) * scale;
    }
}

template <class XT, class AT>
__global__ __launch_bounds__(kThreads) void route_kernel(const XT* __restrict__ x, const AT* __restrict__ w,
                                                         const AT* __restrict__ bias, int64_t T, int h, int E, int k,
                                                         int score, int normalize, AT scale, RouteShape rs,
                                                         AT* __restrict__ logits, int32_t* __restrict__ topi,
                                                         AT* __restrict__ gates) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    AT* part = reinterpret_cast<AT*>(smem_raw);                 // [tb][S][E]
    AT* lg = part + static_cast<size_t>(rs.tb) * rs.S * E;      // [tb][E]
    AT* num = lg + static_cast<size_t>(rs.tb) * E;              // [tb][k]
    int* sel = reinterpret_cast<int*>(num + rs.tb * k);         // [tb][k]

    const int tid = threadIdx.x;
    const int64_t t_block = static_cast<int64_t>(blockIdx.x) * rs.tb;

    // Phase 1: per-segment fused multiply-add chains.
    for (int wi = tid; wi < rs.ntg * rs.units; wi += kThreads) {
        const int tg = wi / rs.units, u = wi % rs.units;
        const int s = u / rs.n_ec, ec = u % rs.n_ec;
        const int e0 = ec * kEpt;
        AT acc[kTpt][kEpt];
#pragma unroll
        for (int a = 0; a < kTpt; ++a)
#pragma unroll
            for (int b = 0; b < kEpt; ++b) acc[a][b] = AT(0);
        const int i_begin = s * rs.seg, i_end = i_begin + rs.seg;
        for (int i = i_begin; i < i_end; i += 8) {
            AT xv[kTpt][8];
#pragma unroll
            for (int a = 0; a < kTpt; ++a) {
                const int64_t t = t_block + tg * kTpt + a;
                if (t < T) {
                    Load8<XT, AT>::run(x + t * h + i, xv[a]);
                } else {
#pragma unroll
                    for (int c = 0; c < 8; ++c) xv[a][c] = AT(0);
                }
            }
#pragma unroll
            for (int b = 0; b < kEpt; ++b) {
                if (e0 + b < E) {
                    AT wv[8];
                    Load8<AT, AT>::run(w + static_cast<int64_t>(e0 + b) * h + i, wv);
#pragma unroll
                    for (int c = 0; c < 8; ++c)
#pragma unroll
                        for (int a = 0; a < kTpt; ++a) acc[a][b] = fma_t(xv[a][c], wv[c], acc[a][b]);
                }
            }
        }
#pragma unroll
        for (int a = 0; a < kTpt; ++a)
#pragma unroll
            for (int b = 0; b < kEpt; ++b)
                if (e0 + b < E) part[(static_cast<size_t>(tg * kTpt + a) * rs.S + s) * E + e0 + b] = acc[a][b];
    }
    __syncthreads();

    // Phase 2: segment sums left to right.
    for (int i = tid; i < rs.tb * E; i += kThreads) {
        const int tl = i / E, e = i % E;
        const AT* pp = part + static_cast<size_t>(tl) * rs.S * E + e;
        AT total = pp[0];
        for (int s = 1; s < rs.S; ++s) total = total + pp[static_cast<size_t>(s) * E];
        lg[i] = total;
        const int64_t t = t_block + tl;
        if (t < T) logits[t * E + e] = total;
    }
    __syncthreads();

    select_and_gate<AT>(lg, E, sel, num, t_block, rs.tb, kThreads, T, E, k, score, normalize, scale, bias, topi, gates);
}

// Router logits of bfloat16 and float32 tokens on the matrix cores, the
// production path.  v_mfma_f32_16x16x4_f32 adds its four products one after
// the other, each a correctly rounded fused multiply-add with subnormals
// (compared with fmaf chains bit for bit on random, subnormal, widely spread
// and NaN / infinite inputs).  So the logits are the very chains of
// route_kernel and the oracle, bit for bit.  (The one-k shapes are exact too,
// at a quarter of the rate.)  A wave's task is 16 experts by TI x 16 tokens by
// four 256-element segments, whose chains are independent.
//
// Each wave streams its rows through LDS of its own, 16 elements of every row
// a batch, NB batches deep, with direct HBM -> LDS loads: read straight into
// registers, every lane's 16 bytes were a cache line of their own and the
// loads' address rate bound the kernel.  No barrier until the chains are
// complete; the chains of a round of tasks then meet in LDS (over the staging
// buffers) and are added left to right.
//   Measured (64 experts, 2048 inputs, top 6; a lane per token on the VALU
// before): 64 tokens 144 -> 26 us, 4096 tokens 165 -> 30, 16384 206 -> 96;
// 4096 tokens by 128 experts, top 8: 328 -> 51; 1000 float32 tokens by 8
// experts, 1024 inputs: 99 -> 14.  What bounds it now: up to 4096 tokens the
// chain of one task (256 MFMAs a wave, two waves a SIMD) and the selection.
constexpr int kRtBatch = 16;
typedef float f32x4_route_t __attribute__((ext_vector_type(4)));

// Staged rows of a 64-row tile (16 rows by 4 segments): C chunks of 16 bytes
// a row, chunk c of row p at c ^ (p / (16 / C) mod C), so that the 16 rows of a
// ds_read_b128 hit distinct banks.
template <int C> __device__ __forceinline__ int rt_chunk(int p, int c) { return c ^ ((p / (16 / C)) & (C - 1)); }

template <class XT, int TI, int W, int NB>
__global__ __launch_bounds__(64 * W) void route_mfma_kernel(const XT* __restrict__ x, const float* __restrict__ w,
                                                            const float* __restrict__ bias, int64_t T, int h, int E,
                                                            int k, int score, int normalize, float scale, int seg,
                                                            int S, float* __restrict__ logits,
                                                            int32_t* __restrict__ topi, float* __restrict__ gates) {
    constexpr int TB = 16 * TI;
    constexpr int XC = kRtBatch * static_cast<int>(sizeof(XT)) / 16, WC = kRtBatch * 4 / 16;   // chunks per staged row
    constexpr int kBufBytes = 1024 * (WC + XC * TI), kLoads = WC + XC * TI;
    __shared__ __align__(1024) uint8_t stage[W * NB * kBufBytes];
    static_assert(W * 4 * 16 * TB * 4 <= W * NB * kBufBytes, "a round's chains fit over the staging buffers");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int ld = E | 1;                                   // odd row pitch: no bank conflicts
    float* lg = reinterpret_cast<float*>(smem_raw);         // [TB][ld]
    float* num = lg + TB * ld;                              // [TB][k]
    int* sel = reinterpret_cast<int*>(num + TB * k);        // [TB][k]
    float* part = reinterpret_cast<float*>(stage);          // [tasks][4 segments][16 experts][TB]
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t t_block = static_cast<int64_t>(blockIdx.x) * TB;
    const int tb = static_cast<int>(min<int64_t>(TB, T - t_block));
    const Rsrc rw = make_dma_rsrc(w, static_cast<int64_t>(E) * h * 4);
    const Rsrc rx = make_dma_rsrc(x + t_block * h, static_cast<int64_t>(tb) * h * sizeof(XT));
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(stage)) + wave * NB * kBufBytes;
    const uint8_t* mine = stage + wave * NB * kBufBytes;
    // A round: ge expert tiles by nq segment quads, one task a wave.
    const int n_sq = (S + 3) / 4, n_et = (E + 15) / 16;
    const int nq = min(n_sq, W), ge = max(1, W / n_sq);
    for (int et0 = 0; et0 < n_et; et0 += ge)
        for (int sq0 = 0; sq0 < n_sq; sq0 += nq) {
            const int tasks = min(ge, n_et - et0) * min(nq, n_sq - sq0), n_q = min(nq, n_sq - sq0);
            f32x4_route_t acc[TI][4];   // [token tile][segment]: tokens 4 q .. + 3 of expert r
#pragma unroll
            for (int t = 0; t < TI; ++t)
#pragma unroll
                for (int b = 0; b < 4; ++b) acc[t][b] = f32x4_route_t{};
            if (wave < tasks) {
                const int e0 = (et0 + wave / n_q) * 16, s0 = 4 * (sq0 + wave % n_q);
                // Byte offsets of the pieces this lane loads; rows past the last expert, token or segment
                // repeat a valid one, and their results are dropped.
                uint32_t ow[WC], ox[TI][XC];
#pragma unroll
                for (int j = 0; j < WC; ++j) {
                    const int p = (j * 64 + lane) / WC, c = rt_chunk<WC>(p, lane % WC);
                    ow[j] = (static_cast<uint32_t>(min(e0 + p % 16, E - 1)) * h + min(s0 + p / 16, S - 1) * seg) * 4u + c * 16u;
                }
#pragma unroll
                for (int t = 0; t < TI; ++t)
#pragma unroll
                    for (int j = 0; j < XC; ++j) {
                        const int p = (j * 64 + lane) / XC, c = rt_chunk<XC>(p, lane % XC);
                        ox[t][j] = (static_cast<uint32_t>(min(16 * t + p % 16, tb - 1)) * h + min(s0 + p / 16, S - 1) * seg) *
                                       static_cast<uint32_t>(sizeof(XT)) + c * 16u;
                    }
                auto issue = [&](int b) {   // the loads of batch b into its buffer
                    const uint32_t at = lds0 + (b % NB) * kBufBytes, i = static_cast<uint32_t>(b) * kRtBatch;
#pragma unroll
                    for (int j = 0; j < WC; ++j) dma16(rw, ow[j], i * 4, at + j * 1024);
#pragma unroll
                    for (int t = 0; t < TI; ++t)
#pragma unroll
                        for (int j = 0; j < XC; ++j)
                            dma16(rx, ox[t][j], i * static_cast<uint32_t>(sizeof(XT)), at + (WC + t * XC + j) * 1024);
                };
                const int nb = (seg + kRtBatch - 1) / kRtBatch;
#pragma unroll
                for (int b = 0; b < NB - 1; ++b)
                    if (b < nb) issue(b);
                for (int b = 0; b < nb; ++b) {
                    if (b + NB - 1 < nb) {
                        __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): batch b - 1 has been read from its buffer
                        issue(b + NB - 1);
                        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NB - 1) * kLoads) : "memory");
                    } else if (NB > 2 && b + 1 < nb) {
                        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NB - 2) * kLoads) : "memory");
                    } else {
                        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    }
                    const uint8_t* buf = mine + (b % NB) * kBufBytes;
                    // Lane l holds element 4 i + q of row r of each 16-row tile (rows 16 seg .. + 15 of the
                    // stage).  Every read of the batch is issued before the first MFMA waits for one.
                    float wf[4][4], xf[TI][4][4];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int sg = 0; sg < 4; ++sg) {
                            const int p = 16 * sg + r;
                            wf[i][sg] = *reinterpret_cast<const float*>(buf + (p * WC + rt_chunk<WC>(p, i)) * 16 + 4 * q);
#pragma unroll
                            for (int t = 0; t < TI; ++t) {
                                const uint8_t* xt = buf + (WC + t * XC) * 1024;
                                if constexpr (sizeof(XT) == 2)
                                    xf[t][i][sg] = bf16_to_f32(*reinterpret_cast<const uint16_t*>(
                                        xt + (p * XC + rt_chunk<XC>(p, i / 2)) * 16 + (i % 2) * 8 + 2 * q));
                                else
                                    xf[t][i][sg] =
                                        *reinterpret_cast<const float*>(xt + (p * XC + rt_chunk<XC>(p, i)) * 16 + 4 * q);
                            }
                        }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (i % 2 == 0 && b * kRtBatch + 4 * i >= seg) break;   // a segment shorter than 256 may end here
#pragma unroll
                        for (int sg = 0; sg < 4; ++sg)
#pragma unroll
                            for (int t = 0; t < TI; ++t)
                                acc[t][sg] = __builtin_amdgcn_mfma_f32_16x16x4f32(xf[t][i][sg], wf[i][sg], acc[t][sg], 0, 0, 0);
                    }
                }
            }
            __syncthreads();   // every wave is done with its staging buffers
            if (wave < tasks)
#pragma unroll
                for (int b = 0; b < 4; ++b)
#pragma unroll
                    for (int t = 0; t < TI; ++t)
                        *reinterpret_cast<float4*>(part + ((wave * 4 + b) * 16 + r) * TB + 16 * t + 4 * q) =
                            make_float4(acc[t][b][0], acc[t][b][1], acc[t][b][2], acc[t][b][3]);
            __syncthreads();
            const int s_end = min(4 * n_q, S - 4 * sq0);   // segments of this round
            for (int idx = threadIdx.x; idx < min(ge, n_et - et0) * 16 * TB; idx += 64 * W) {
                const int tile = idx / (16 * TB), at = idx % (16 * TB), e = (et0 + tile) * 16 + at / TB;
                if (e < E) {
                    const float* pp = part + tile * n_q * 4 * 16 * TB + at;
                    float* out = lg + (at % TB) * ld + e;
                    float total = sq0 ? *out + pp[0] : pp[0];
                    for (int s = 1; s < s_end; ++s) total = total + pp[s * 16 * TB];
                    *out = total;
                }
            }
            __syncthreads();   // the sums are read before the next round's loads land
        }
    for (int idx = threadIdx.x; idx < tb * E; idx += 64 * W) logits[t_block * E + idx] = lg[(idx / E) * ld + idx % E];
    select_and_gate<float>(lg, ld, sel, num, t_block, TB, 64 * W, T, E, k, score, normalize, scale, bias, topi, gates);
}

}  // namespace

// ---------------------------------------------------------------------------- dispatch plan

namespace {

constexpr int kDispatchPairs = 4096;   // pairs per dispatch block (upper bound)

struct DispatchShape {
    int64_t T;
    int k, E, e0, e1, n_src, tokens_per_block, nblk;
};

// Token range [ts, te) and source of dispatch block b; blocks never straddle sources.
__device__ __forceinline__ void block_range(const DispatchShape& d, int b, int64_t* ts, int64_t* te, int* src) {
    const int64_t base = d.T / d.n_src, rem = d.T % d.n_src;
    int64_t start = 0;
    for (int s = 0; s < d.n_src; ++s) {
        const int64_t len = base + (s < rem ? 1 : 0);
        const int64_t nb = (len + d.tokens_per_block - 1) / d.tokens_per_block;
        if (b < nb) {
            *ts = start + static_cast<int64_t>(b) * d.tokens_per_block;
            *te = std::min(*ts + d.tokens_per_block, start + len);
            *src = s;
            return;
        }
        b -= static_cast<int>(nb);
        start += len;
    }
    *ts = *te = 0;
    *src = -1;
}

__device__ __forceinline__ uint64_t lanemask_lt(int lane) { return (lane == 0) ? 0ull : ((~0ull) >> (64 - lane)); }

// Lanes of the wave whose key equals mine (among lanes with valid keys), in
// nbits ballots: a lane matches when it agrees with mine on every key bit.
// Keys lie in [0, 2^nbits).
__device__ __forceinline__ uint64_t match_any(bool valid, int key, int nbits) {
    uint64_t m = __ballot(valid);
    for (int i = 0; i < nbits; ++i) {
        const bool bit = (key >> i) & 1;
        const uint64_t b = __ballot(valid && bit);
        m &= bit ? b : ~b;
    }
    return valid ? m : 0ull;
}

// Bits of the largest key n - 1 (at least one).
__host__ __device__ constexpr int key_bits(int n) {
    int b = 1;
    while ((1 << b) < n) ++b;
    return b;
}

constexpr int kDispatchRounds = kDispatchPairs / kThreads;   // rounds of one pair per thread in a block

// The expert ids of a block's pairs, loaded all at once (one pair per thread
// and round, pair p0 + r kThreads + thread): every round's load is in flight
// together, not one at a time.  Entries past the block are not read.
__device__ __forceinline__ void load_block_ids(const int32_t* topi, int64_t p0, int64_t p1,
                                               int (&e)[kDispatchRounds]) {
#pragma unroll
    for (int r = 0; r < kDispatchRounds; ++r) {
        const int64_t p = p0 + static_cast<int64_t>(r) * kThreads + threadIdx.x;
        e[r] = p < p1 ? topi[p] : 0;
    }
}

// The whole plan of one source's at most kDispatchPairs pairs in one block, in
// place of the three kernels below: with so few pairs they are launch latency
// (kernel time, 8 tokens by 2 slots, 8 experts: 10.5 us in three launches, 3.2 in
// one; 64 by 6, 64 experts: 17.3 and 5.1; 2048 by 2, 8 experts: 19.3 and 13.3;
// 512 by 8, 128 experts: 27.1 and 20.0).  Wave w
// takes the w-th quarter of the pairs, in order, so ranks need no exchange
// between waves beyond one scan: it counts its pairs per expert, the block
// turns the counts into each wave's first place within each expert and the
// experts' first rows, and each wave then places its pairs, 64 at a time.
// More pairs keep the kernels below, whose blocks share the work.  256 threads
// for the reason given at dispatch_scan_kernel.
__global__ __launch_bounds__(kThreads) void dispatch_one_block_kernel(const int32_t* __restrict__ topi, DispatchShape d,
                                                                      int32_t* __restrict__ counts,
                                                                      int32_t* __restrict__ offsets,
                                                                      int32_t* __restrict__ src_counts,
                                                                      int32_t* __restrict__ perm,
                                                                      int32_t* __restrict__ pair_row) {
    constexpr int kWaves = kThreads / 64, kRounds = kDispatchPairs / kThreads;
    __shared__ int place[kWaves][kMaxE + 1];   // pairs of (wave, expert), then the next place in the expert
    __shared__ int tot[kMaxE + 1];
    __shared__ int off[kMaxE];
    const int L = d.e1 - d.e0;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int P = static_cast<int>(d.T) * d.k;
    const int rounds = (P + kThreads - 1) / kThreads, p0 = wave * rounds * 64 + lane;
    int ids[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        const int p = p0 + r * 64;
        const int e = r < rounds && p < P ? topi[p] : -1;
        ids[r] = e < 0 || e >= d.E ? d.E : e;   // d.E counts ids outside [0, E)
    }
    for (int e = lane; e <= d.E; e += 64) place[wave][e] = 0;
    const int nbits = key_bits(d.E + 1);
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        if (r >= rounds) break;
        const uint64_t m = match_any(p0 + r * 64 < P, ids[r], nbits);
        if (m && (m & lanemask_lt(lane)) == 0) atomicAdd(&place[wave][ids[r]], __popcll(m));
    }
    __syncthreads();
    for (int e = threadIdx.x; e <= d.E; e += kThreads) {
        int sum = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const int c = place[w][e];
            place[w][e] = sum;
            sum += c;
        }
        tot[e] = sum;
        counts[e] = sum;
    }
    __syncthreads();
    if (wave == 0) {   // the local experts' first rows, 64 experts at a time
        int run = 0;
        for (int i0 = 0; i0 < L; i0 += 64) {
            const int i = i0 + lane, c = i < L ? tot[d.e0 + i] : 0;
            int incl = c;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int up = __shfl_up(incl, o, 64);
                if (lane >= o) incl += up;
            }
            if (i < L) {
                off[i] = run + incl - c;
                offsets[i] = run + incl - c;
                src_counts[i] = c;
            }
            run += __shfl(incl, 63, 64);
        }
        if (lane == 0) offsets[L] = run;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        if (r >= rounds) break;
        const int p = p0 + r * 64, e = ids[r];
        const bool local = p < P && e >= d.e0 && e < d.e1;
        const uint64_t m = match_any(local, e, nbits);
        const int rank = __popcll(m & lanemask_lt(lane));
        int first = 0;
        if (local && rank == 0) first = off[e - d.e0] + atomicAdd(&place[wave][e], __popcll(m));
        first = __shfl(first, local ? __ffsll(static_cast<unsigned long long>(m)) - 1 : lane, 64);
        if (local) {
            perm[first + rank] = p;
            pair_row[p] = first + rank;
        } else if (p < P) {
            pair_row[p] = -1;
        }
    }
}

// Phase 1: per-block expert histogram; one LDS atomic per distinct id of a wave and round.
__global__ __launch_bounds__(kThreads) void dispatch_count_kernel(const int32_t* __restrict__ topi, DispatchShape d,
                                                                  int32_t* __restrict__ block_counts,
                                                                  int32_t* __restrict__ block_src) {
    __shared__ int hist[kMaxE + 1];
    const int b = blockIdx.x;
    for (int e = threadIdx.x; e <= d.E; e += kThreads) hist[e] = 0;
    int64_t ts, te;
    int src;
    block_range(d, b, &ts, &te, &src);
    int ids[kDispatchRounds];
    load_block_ids(topi, ts * d.k, te * d.k, ids);
    __syncthreads();
    const int lane = threadIdx.x & 63, nbits = key_bits(d.E + 1);
    const int64_t p0 = ts * d.k, p1 = te * d.k;
#pragma unroll
    for (int r = 0; r < kDispatchRounds; ++r) {
        const bool valid = p0 + static_cast<int64_t>(r) * kThreads + threadIdx.x < p1;
        const int e = ids[r] < 0 || ids[r] >= d.E ? d.E : ids[r];   // d.E counts ids outside [0, E)
        const uint64_t m = match_any(valid, e, nbits);
        if (valid && (m & lanemask_lt(lane)) == 0) atomicAdd(&hist[e], __popcll(m));
    }
    __syncthreads();
    for (int e = threadIdx.x; e <= d.E; e += kThreads) block_counts[static_cast<int64_t>(b) * (d.E + 1) + e] = hist[e];
    if (threadIdx.x == 0) block_src[b] = src;
}

// Phase 2 (one block): totals, local offsets, per-source counts and the base
// row of every (block, local expert).  The per-block histograms are staged in
// LDS first (one load per entry, all in flight together) when they fit.
// Two sizes: up to 255 experts and 8192 staged entries, a 256-thread block
// with 38 KB of LDS; beyond that, 1024 threads and 88 KB.  The small block
// matters where the plan runs beside a kernel that fills every CU with small
// blocks (the fp8 weight cast): a 1024-thread block waits for 16 free wave
// slots on one CU, which that kernel's blocks take first, and the plan's
// next kernels wait behind it.
template <int NT, int MAXE, int STAGE, int STAGE_SRC>
__global__ __launch_bounds__(NT) void dispatch_scan_kernel(const int32_t* __restrict__ block_counts,
                                                           const int32_t* __restrict__ block_src, DispatchShape d,
                                                           int32_t* __restrict__ counts,
                                                           int32_t* __restrict__ offsets,
                                                           int32_t* __restrict__ src_counts,
                                                           int32_t* __restrict__ block_base) {
    __shared__ int tot[MAXE + 1];
    __shared__ int off[MAXE + 1];
    __shared__ int stage[STAGE];
    __shared__ int stage_src[STAGE_SRC];
    const int L = d.e1 - d.e0, W = d.E + 1;
    const int64_t n = static_cast<int64_t>(d.nblk) * W;
    const bool staged = n <= STAGE, staged_src = d.nblk <= STAGE_SRC;
    if (staged)
        for (int i = threadIdx.x; i < n; i += blockDim.x) stage[i] = block_counts[i];
    if (staged_src)
        for (int i = threadIdx.x; i < d.nblk; i += blockDim.x) stage_src[i] = block_src[i];
    __syncthreads();
    auto cnt = [&](int b, int e) { return staged ? stage[b * W + e] : block_counts[static_cast<int64_t>(b) * W + e]; };
    auto src_of = [&](int b) { return staged_src ? stage_src[b] : block_src[b]; };
    for (int e = threadIdx.x; e <= d.E; e += blockDim.x) {
        int sum = 0;
        for (int b = 0; b < d.nblk; ++b) sum += cnt(b, e);
        tot[e] = sum;
        counts[e] = sum;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int run = 0;
        for (int i = 0; i < L; ++i) {
            off[i] = run;
            offsets[i] = run;
            run += tot[d.e0 + i];
        }
        off[L] = run;
        offsets[L] = run;
    }
    for (int i = threadIdx.x; i < d.n_src * L; i += blockDim.x) src_counts[i] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < L; i += blockDim.x) {
        const int e = d.e0 + i;
        int run = off[i];
        int cur_src = -1, cur = 0;
        for (int b = 0; b < d.nblk; ++b) {
            const int c = cnt(b, e);
            block_base[static_cast<int64_t>(b) * L + i] = run;
            run += c;
            const int s = src_of(b);
            if (s != cur_src) {
                if (cur_src >= 0) src_counts[cur_src * L + i] = cur;
                cur_src = s;
                cur = 0;
            }
            cur += c;
        }
        if (cur_src >= 0) src_counts[cur_src * L + i] = cur;
    }
}

// Phase 3: stable scatter.  Pairs of a block are ranked in ascending p: within
// a wave by lane order, across the block's waves by wave order, across
// rounds by a running per-expert count.
__global__ __launch_bounds__(kThreads) void dispatch_scatter_kernel(const int32_t* __restrict__ topi, DispatchShape d,
                                                                    const int32_t* __restrict__ block_base,
                                                                    int32_t* __restrict__ perm,
                                                                    int32_t* __restrict__ pair_row) {
    __shared__ int wcnt[kThreads / 64][kMaxE];
    __shared__ int run[kMaxE];
    const int L = d.e1 - d.e0;
    const int b = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < L; i += kThreads) {
        run[i] = block_base[static_cast<int64_t>(b) * L + i];
#pragma unroll
        for (int w = 0; w < kThreads / 64; ++w) wcnt[w][i] = 0;
    }
    int64_t ts, te;
    int src;
    block_range(d, b, &ts, &te, &src);
    const int64_t p0 = ts * d.k, p1 = te * d.k;
    int ids[kDispatchRounds];
    load_block_ids(topi, p0, p1, ids);
    __syncthreads();
    const int nbits = key_bits(L);
    for (int r = 0; r < kDispatchRounds; ++r) {
        const int64_t p = p0 + static_cast<int64_t>(r) * kThreads + threadIdx.x;
        if (p0 + static_cast<int64_t>(r) * kThreads >= p1) break;   // uniform: no pairs left in the block
        const bool in = p < p1;
        const int e = ids[r];
        const bool local = in && e >= d.e0 && e < d.e1;
        const int li = local ? e - d.e0 : 0;
        const uint64_t m = match_any(local, li, nbits);
        const int rank = __popcll(m & lanemask_lt(lane));
        if (local && rank == 0) wcnt[wave][li] = __popcll(m);
        __syncthreads();
        if (local) {
            int pre = run[li];
            for (int w = 0; w < wave; ++w) pre += wcnt[w][li];
            const int row = pre + rank;
            perm[row] = static_cast<int32_t>(p);
            pair_row[p] = row;
        } else if (in) {
            pair_row[p] = -1;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < L; i += kThreads) {
            int add = 0;
#pragma unroll
            for (int w = 0; w < kThreads / 64; ++w) {
                add += wcnt[w][i];
                wcnt[w][i] = 0;
            }
            run[i] += add;
        }
        __syncthreads();
    }
}

int dispatch_blocks(int64_t T, int k, int n_src, int* tokens_per_block) {
    const int tpb = std::max(1, kDispatchPairs / k);
    *tokens_per_block = tpb;
    const int64_t base = T / n_src, rem = T % n_src;
    int64_t nb = 0;
    for (int s = 0; s < n_src; ++s) {
        const int64_t len = base + (s < rem ? 1 : 0);
        nb += (len + tpb - 1) / tpb;
    }
    return static_cast<int>(nb);
}

// ---------------------------------------------------------------------------- bias update, route backward

template <class AT>
__global__ void bias_update_kernel(AT* bias, const int32_t* counts, int E, AT rate) {
    __shared__ long long total;
    if (threadIdx.x == 0) {
        long long s = 0;
        for (int e = 0; e < E; ++e) s += counts[e];
        total = s;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
        // sign(mean - load) == sign(sum - E * load), evaluated exactly in integers.
        const long long diff = total - static_cast<long long>(E) * counts[e];
        const AT sgn = diff > 0 ? AT(1) : (diff < 0 ? AT(-1) : AT(0));
        bias[e] = bias[e] + rate * sgn;
    }
}

template <class AT>
__global__ __launch_bounds__(kThreads) void route_bwd_kernel(const AT* __restrict__ dgates,
                                                             const AT* __restrict__ gates,
                                                             const AT* __restrict__ logits,
                                                             const int32_t* __restrict__ topi, int64_t T, int E, int k,
                                                             int score, int normalize, AT scale,
                                                             AT* __restrict__ dl) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= T) return;
    const AT* g = gates + t * k;
    const AT* dg = dgates + t * k;
    AT dot = AT(0);
    for (int j = 0; j < k; ++j) dot = dot + g[j] * dg[j];
    if (score == RHP_SCORE_SOFTMAX) {
        // g = c * softmax(l_sel):  dl_i = g_i * (dg_i - sum_j g_j dg_j / c)
        const AT corr = dot / scale;
        for (int j = 0; j < k; ++j) dl[t * k + j] = g[j] * (dg[j] - corr);
    } else {
        AT ssum = AT(0);
        AT s[kMaxTopK];
        for (int j = 0; j < k; ++j) {
            const int e = topi[t * k + j];
            s[j] = (e >= 0 && e < E) ? rhp_sigmoid(logits[t * E + e]) : AT(0);
            ssum = ssum + s[j];
        }
        for (int j = 0; j < k; ++j) {
            // normalised: g = c s / S  ->  ds_i = (c / S) (dg_i - sum_j g_j dg_j / c);  else ds = c dg
            const AT ds = normalize ? (scale / ssum) * (dg[j] - dot / scale) : scale * dg[j];
            dl[t * k + j] = ds * s[j] * (AT(1) - s[j]);
        }
    }
}

// LDS of a route_mfma_kernel block beside its staging buffers (logits and selection of its tokens), and
// what the buffers of eight waves leave for it.
constexpr size_t rt_lds(int tb, int E, int k) { return static_cast<size_t>(tb) * ((E | 1) + 2 * k) * 4; }
template <class XT, int TI, int NB> constexpr size_t rt_room() {
    return 163840 - 8 * NB * 1024 * (kRtBatch * 4 / 16 + kRtBatch * sizeof(XT) / 16 * TI);
}
// bfloat16 tokens from which a block takes 32: they stage the weights half as often, but 16-token blocks
// are quicker until they fill the CUs twice (64 experts: 4096 tokens 37 against 54 us, 8192 both 57).
constexpr int64_t kRtWideTokens = 8192;

template <class XT, int TI, int NB>
int launch_route_mfma(const void* x, const void* w, const void* bias, int64_t T, int h, int E, int k, int score,
                      int normalize, double scale, void* logits, int32_t* topi, void* gates, hipStream_t stream) {
    const int seg = std::min(256, h), S = h / seg, tasks = ((E + 15) / 16) * ((S + 3) / 4);
    auto go = [&](auto kern, int waves) {
        hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>((T + 16 * TI - 1) / (16 * TI))), dim3(64 * waves),
                           rt_lds(16 * TI, E, k), stream, static_cast<const XT*>(x), static_cast<const float*>(w),
                           static_cast<const float*>(bias), T, h, E, k, score, normalize, static_cast<float>(scale),
                           seg, S, static_cast<float*>(logits), topi, static_cast<float*>(gates));
    };
    if (tasks <= 4) go(route_mfma_kernel<XT, TI, 4, NB>, 4);
    else go(route_mfma_kernel<XT, TI, 8, NB>, 8);
    return check_launch("route_mfma_kernel");
}

// Sizes a route_mfma_kernel takes, whatever the token count: its block's logits and selection fit beside the
// staging buffers, and the byte offsets of the router's and of a block's token rows in 31 bits.
template <class XT, int TI, int NB> bool rt_takes(int h, int E, int k) {
    constexpr int64_t limit = int64_t(1) << 31;
    return rt_lds(16 * TI, E, k) <= rt_room<XT, TI, NB>() && static_cast<int64_t>(E) * h * 4 < limit &&
           int64_t(16) * TI * h * static_cast<int64_t>(sizeof(XT)) < limit;
}

template <class XT, class AT>
int launch_route(const void* x, const void* w, const void* bias, int64_t T, int h, int E, int k, int score,
                 int normalize, double scale, void* logits, int32_t* topi, void* gates, hipStream_t stream) {
    if constexpr (std::is_same<AT, float>::value) {
        int (*mfma)(const void*, const void*, const void*, int64_t, int, int, int, int, int, double, void*, int32_t*,
                    void*, hipStream_t) = nullptr;
        if constexpr (std::is_same<XT, bf16>::value) {
            if (T >= kRtWideTokens && rt_takes<XT, 2, 2>(h, E, k)) mfma = launch_route_mfma<XT, 2, 2>;
            else if (rt_takes<XT, 1, 3>(h, E, k)) mfma = launch_route_mfma<XT, 1, 3>;
        }
        if (!mfma && rt_takes<XT, 1, 2>(h, E, k)) mfma = launch_route_mfma<XT, 1, 2>;
        if (mfma) {
            if (T == 0) return 0;
            return mfma(x, w, bias, T, h, E, k, score, normalize, scale, logits, topi, gates, stream);
        }
    }
    // float64 tokens, and more experts than the kernel above holds (E + 2 k past 1023 in bfloat16, 511 in float32).
    RouteShape rs;
    rs.seg = std::min(256, h);
    rs.S = h / rs.seg;
    rs.n_ec = (E + kEpt - 1) / kEpt;
    rs.units = rs.S * rs.n_ec;
    // Tokens per block: as many token groups as fill the block, capped so the
    // per-block partial sums fit in 48 KiB of LDS.
    int ntg = std::max(1, kThreads / rs.units);
    const size_t per_token = (static_cast<size_t>(rs.S) * E + E) * sizeof(AT) + static_cast<size_t>(k) * sizeof(int);
    while (ntg > 1 && static_cast<size_t>(ntg) * kTpt * per_token > 48 * 1024) --ntg;
    rs.ntg = ntg;
    rs.tb = ntg * kTpt;
    const size_t smem = static_cast<size_t>(rs.tb) * per_token;
    RHP_REQUIRE(smem <= 48 * 1024, "rhp_route: hidden size x experts too large for one routing block");
    if (T == 0) return 0;
    const int64_t blocks = (T + rs.tb - 1) / rs.tb;
    hipLaunchKernelGGL((route_kernel<XT, AT>), dim3(static_cast<unsigned>(blocks)), dim3(kThreads),
                       smem + static_cast<size_t>(rs.tb) * k * sizeof(AT), stream,
                       static_cast<const XT*>(x), static_cast<const AT*>(w), static_cast<const AT*>(bias), T, h, E, k,
                       score, normalize, static_cast<AT>(scale), rs, static_cast<AT*>(logits), topi,
                       static_cast<AT*>(gates));
    return check_launch("route_kernel");
}

}  // namespace
}  // namespace rhp

using namespace rhp;

extern "C" int rhp_route(const void* x, int x_dtype, const void* router_w, int r_dtype, const void* bias, int64_t T,
                         int h, int E, int k, int score, int normalize, double scale, void* logits, int32_t* topi,
                         void* gates, hipStream_t stream) {
    clear_error();
    RHP_REQUIRE(T >= 0 && h > 0 && E > 0, "rhp_route: T must be >= 0 and h, E > 0");
    RHP_REQUIRE(h % 8 == 0 && h % std::min(256, h) == 0, "rhp_route: h must be a multiple of 8 and of min(256, h)");
    RHP_REQUIRE(E <= kMaxE, "rhp_route: at most 1024 experts");
    RHP_REQUIRE(k >= 1 && k <= E && k <= kMaxTopK, "rhp_route: need 1 <= k <= min(E, 16)");
    RHP_REQUIRE(score == RHP_SCORE_SOFTMAX || score == RHP_SCORE_SIGMOID, "rhp_route: unknown score function");
    RHP_REQUIRE(T == 0 || (x && router_w && logits && topi && gates), "rhp_route: null pointer");
    RHP_REQUIRE(T == 0 || (aligned16(x) && aligned16(router_w)), "rhp_route: x and router_w must be 16-byte aligned");
    if (x_dtype == RHP_F64) {
        RHP_REQUIRE(r_dtype == RHP_F64, "rhp_route: a float64 model needs a float64 router");
        return launch_route<double, double>(x, router_w, bias, T, h, E, k, score, normalize, scale, logits, topi,
                                            gates, stream);
    }
    RHP_REQUIRE(r_dtype == RHP_F32, "rhp_route: float32 / bfloat16 models need a float32 router");
    if (x_dtype == RHP_F32)
        return launch_route<float, float>(x, router_w, bias, T, h, E, k, score, normalize, scale, logits, topi, gates,
                                          stream);
    if (x_dtype == RHP_BF16)
        return launch_route<bf16, float>(x, router_w, bias, T, h, E, k, score, normalize, scale, logits, topi, gates,
                                         stream);
    return fail(std::string("rhp_route: unsupported x dtype ") + dtype_name(x_dtype));
}

extern "C" size_t rhp_dispatch_workspace_bytes(int64_t T, int k, int E, int n_src) {
    if (T < 0 || k <= 0 || E <= 0 || n_src <= 0) return 0;
    int tpb;
    const int nblk = dispatch_blocks(T, k, n_src, &tpb);
    // block_counts [nblk][E+1], block_base [nblk][E], block_src [nblk]
    return static_cast<size_t>(nblk) * (2 * static_cast<size_t>(E) + 2) * sizeof(int32_t) + 256;
}

namespace rhp {
namespace {

// The dispatch plan with its workspace: argument checks, then the one-block
// kernel (few pairs of one source) or the count, scan and scatter kernels.  Every launch writes each workspace entry it
// reads (per-block histograms, sources and base rows), so the workspace
// needs no clearing.
int dispatch_run(const char* fn, const int32_t* topi, int64_t T, int k, int E, int e0, int e1, int n_src,
                 int32_t* counts, int32_t* offsets, int32_t* src_counts, int32_t* perm, int32_t* pair_row,
                 void* workspace, size_t workspace_bytes, hipStream_t stream) {
    const std::string f(fn);
    RHP_REQUIRE(T >= 0 && k >= 1 && E >= 1 && E <= kMaxE, f + ": need T >= 0, k >= 1, 1 <= E <= 1024");
    RHP_REQUIRE(0 <= e0 && e0 < e1 && e1 <= E, f + ": need 0 <= e0 < e1 <= E");
    RHP_REQUIRE(n_src >= 1 && n_src <= (1 << 20), f + ": need 1 <= n_src <= 2^20");
    RHP_REQUIRE(T * k < (int64_t(1) << 31), f + ": T * k must fit in int32");
    RHP_REQUIRE(workspace_bytes >= rhp_dispatch_workspace_bytes(T, k, E, n_src),
                f + ": workspace smaller than rhp_dispatch_workspace_bytes()");
    RHP_REQUIRE(counts && offsets && src_counts && workspace, f + ": null pointer");
    RHP_REQUIRE(T == 0 || (topi && perm && pair_row), f + ": null pointer");
    DispatchShape d;
    d.T = T;
    d.k = k;
    d.E = E;
    d.e0 = e0;
    d.e1 = e1;
    d.n_src = n_src;
    d.nblk = dispatch_blocks(T, k, n_src, &d.tokens_per_block);
    if (n_src == 1 && T > 0 && T * k <= kDispatchPairs) {
        hipLaunchKernelGGL(dispatch_one_block_kernel, dim3(1), dim3(kThreads), 0, stream, topi, d, counts, offsets,
                           src_counts, perm, pair_row);
        return check_launch("dispatch_one_block_kernel");
    }
    const int L = e1 - e0;
    int32_t* block_counts = static_cast<int32_t*>(workspace);
    int32_t* block_base = block_counts + static_cast<size_t>(d.nblk) * (E + 1);
    int32_t* block_src = block_base + static_cast<size_t>(d.nblk) * L;
    if (d.nblk > 0) {
        hipLaunchKernelGGL(dispatch_count_kernel, dim3(d.nblk), dim3(kThreads), 0, stream, topi, d, block_counts,
                           block_src);
        if (int rc = check_launch("dispatch_count_kernel")) return rc;
    }
    if (E + 1 <= 256 && static_cast<int64_t>(d.nblk) * (E + 1) <= 8192)
        hipLaunchKernelGGL((dispatch_scan_kernel<256, 255, 8192, 1024>), dim3(1), dim3(256), 0, stream, block_counts,
                           block_src, d, counts, offsets, src_counts, block_base);
    else
        hipLaunchKernelGGL((dispatch_scan_kernel<1024, kMaxE, 16384, 4096>), dim3(1), dim3(1024), 0, stream,
                           block_counts, block_src, d, counts, offsets, src_counts, block_base);
    if (int rc = check_launch("dispatch_scan_kernel")) return rc;
    if (d.nblk > 0) {
        hipLaunchKernelGGL(dispatch_scatter_kernel, dim3(d.nblk), dim3(kThreads), 0, stream, topi, d, block_base,
                           perm, pair_row);
        if (int rc = check_launch("dispatch_scatter_kernel")) return rc;
    }
    return 0;
}

}  // namespace
}  // namespace rhp

extern "C" int rhp_dispatch(const int32_t* topi, int64_t T, int k, int E, int e0, int e1, int n_src,
                            int32_t* counts, int32_t* offsets, int32_t* src_counts, int32_t* perm, int32_t* pair_row,
                            void* workspace, size_t workspace_bytes, hipStream_t stream) {
    clear_error();
    return dispatch_run("rhp_dispatch", topi, T, k, E, e0, e1, n_src, counts, offsets, src_counts, perm, pair_row,
                        workspace, workspace_bytes, stream);
}

// ---------------------------------------------------------------------------- dispatch without allocation

// The workspace of rhp_dispatch_noalloc: a fixed device array, one per GPU,
// held until the process ends.  In host code its name is not a device
// address; the address comes from hipGetSymbolAddress, once per device.
constexpr size_t kScratchBytes = size_t(4) << 20;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

namespace rhp {
namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of this GPU's scratch array (the current device's).
int scratch_of_current_device(const char* fn, void** out) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
        return fail(std::string(fn) + ": no current HIP device");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || p == nullptr)
            return fail(std::string(fn) + ": hipGetSymbolAddress of the scratch array failed: " + hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return 0;
}

}  // namespace
}  // namespace rhp

extern "C" int rhp_dispatch_noalloc(const int32_t* topi, int64_t T, int k, int E, int e0, int e1, int n_src,
                                    int32_t* counts, int32_t* offsets, int32_t* src_counts, int32_t* perm,
                                    int32_t* pair_row, hipStream_t stream) {
    clear_error();
    RHP_REQUIRE(T >= 0 && k >= 1 && E >= 1 && n_src >= 1, "rhp_dispatch_noalloc: need T >= 0, k >= 1, E >= 1, n_src >= 1");
    const size_t need = rhp_dispatch_workspace_bytes(T, k, E, n_src);
    RHP_REQUIRE(need <= kScratchBytes, "rhp_dispatch_noalloc: these sizes need " + std::to_string(need) +
                                           " bytes of scratch, more than the library's 4 MiB; use rhp_dispatch");
    void* ws = nullptr;
    if (int rc = scratch_of_current_device("rhp_dispatch_noalloc", &ws)) return rc;
    return dispatch_run("rhp_dispatch_noalloc", topi, T, k, E, e0, e1, n_src, counts, offsets, src_counts, perm,
                        pair_row, ws, kScratchBytes, stream);
}

extern "C" int rhp_update_expert_bias(void* bias, int r_dtype, const int32_t* counts, int E, double rate,
                                      hipStream_t stream) {
    clear_error();
    RHP_REQUIRE(bias && counts && E >= 1 && E <= kMaxE, "rhp_update_expert_bias: bad arguments");
    if (r_dtype == RHP_F64) {
        hipLaunchKernelGGL(bias_update_kernel<double>, dim3(1), dim3(256), 0, stream, static_cast<double*>(bias),
                           counts, E, rate);
    } else if (r_dtype == RHP_F32) {
        hipLaunchKernelGGL(bias_update_kernel<float>, dim3(1), dim3(256), 0, stream, static_cast<float*>(bias),
                           counts, E, static_cast<float>(rate));
    } else {
        return fail("rhp_update_expert_bias: bias must be float32 or float64");
    }
    return check_launch("bias_update_kernel");
}

extern "C" int rhp_route_bwd(const void* dgates, const void* gates, const void* logits, const int32_t* topi,
                             int r_dtype, int64_t T, int E, int k, int score, int normalize, double scale,
                             void* dlogits_sel, hipStream_t stream) {
    clear_error();
    RHP_REQUIRE(T >= 0 && E >= 1 && k >= 1 && k <= E && k <= kMaxTopK, "rhp_route_bwd: bad sizes");
    RHP_REQUIRE(scale != 0.0, "rhp_route_bwd: scale must be nonzero");
    if (T == 0) return 0;
    RHP_REQUIRE(dgates && gates && logits && topi && dlogits_sel, "rhp_route_bwd: null pointer");
    const unsigned blocks = static_cast<unsigned>((T + kThreads - 1) / kThreads);
    if (r_dtype == RHP_F64) {
        hipLaunchKernelGGL(route_bwd_kernel<double>, dim3(blocks), dim3(kThreads), 0, stream,
                           static_cast<const double*>(dgates), static_cast<const double*>(gates),
                           static_cast<const double*>(logits), topi, T, E, k, score, normalize, scale,
                           static_cast<double*>(dlogits_sel));
    } else if (r_dtype == RHP_F32) {
        hipLaunchKernelGGL(route_bwd_kernel<float>, dim3(blocks), dim3(kThreads), 0, stream,
                           static_cast<const float*>(dgates), static_cast<const float*>(gates),
                           static_cast<const float*>(logits), topi, T, E, k, score, normalize,
                           static_cast<float>(scale), static_cast<float*>(dlogits_sel));
    } else {
        return fail("rhp_route_bwd: router dtype must be float32 or float64");
    }
    return check_launch("route_bwd_kernel");
}
