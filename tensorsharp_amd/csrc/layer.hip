// Single-token attention pieces of the whole-layer decode (TensorSharp.GGML.Native/ggml_ops_transformer.cpp:318-470):
// what sits between the fused QKV projection and the output projection.
//
//   attn_decode_kernel   first finishes the projections for the heads it serves - optional RMSNorm over the head
//                        (ggml_rms_norm, then * weight), RoPE at `position` (ggml_rope_ext with n_dims = head_dim,
//                        ext_factor 0, attn_factor 1: ggml-cpu/ops.cpp:5549-5563, :5636-5652); the new k and the
//                        untouched v row go into the fp32 KV cache [kv_head][max_seq_len][head_dim] at row `position`
//                        (written by the workgroup of the last split, which uses them from LDS) - then computes
//                        softmax(q . K^T / sqrt(head_dim)) V over positions 0..position (what ggml_flash_attn_ext
//                        computes for one query row); a workgroup serves the query heads that share a KV head, so K / V
//                        rows are loaded once per group; the positions are cut into splits of 64 or 128 (attn_rows), each split
//                        leaves (max, sum, weighted V) behind (a single split writes the result itself)
//   attn_combine_kernel  merges the splits of a head
//
// HBM-bound on the KV cache: 2 * num_kv_heads * (position + 1) * head_dim * 4 bytes per call.
#include "tship_internal.h"

#include <algorithm>

namespace tship {
namespace {

constexpr int kMaxHeadDim = 256;
constexpr int kAttnWaves = 8;
constexpr int kAttnGroups = 4 * kAttnWaves;      // 16-lane groups of a workgroup
// K / V rows per 16-lane group, all requested at once; a workgroup's split is kAttnGroups times as many positions.  The kernel
// is latency bound: two rows (more and shorter workgroups) while every CU has at most one workgroup per KV head's split and the
// merge takes one batch of 64 splits, four beyond and where that leaves a single split and no merge.  Measured us per small
// layer, two / four rows (query x KV heads): 32 x 8 64 positions 22.7 / 23.7, 100 25.2 / 23.6, 512 25.2 / 26.3, 2048 27.7 / 28.4,
// 3000 32.0 / 30.8; 8 x 2 4001 24.8 / 26.2, 8192 27.7 / 27.2; 16 x 2 6000 29.1 / 26.9; 32 x 32 512 26.8 / 27.4, 700 29.8 / 29.4.
// One query head per KV head takes two rows somewhat longer, its small workgroups fit four to a CU (two small layers, two / four
// rows: 32 x 32 heads at 2049 positions 66.8 / 69.6, 2400 68.2 / 69.7, 2600 71.2 / 70.4, 16 x 16 at 2049 53.7 / 56.5, 2400 54.3 / 56.3).
constexpr int kFewSplits = 64, kFewSplitsOneHead = 40;
int attn_rows(int num_heads, int num_kv_heads, int total)
{
    if (total <= 2 * kAttnGroups) return 2;
    if (total <= 4 * kAttnGroups) return 4;
    const int splits = (total + 2 * kAttnGroups - 1) / (2 * kAttnGroups);
    if (num_heads == num_kv_heads && splits <= kFewSplitsOneHead) return 2;
    return splits <= kFewSplits && (int64_t)num_kv_heads * splits <= device_info().num_cus ? 2 : 4;
}

__device__ __forceinline__ float wave_sum(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}
// (register permutations on both halves of the value; a shuffle of a double is two trips through the LDS crossbar)
__device__ __forceinline__ double wave_sum(double v)
{
    typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
    auto moved = [](double d, auto perm) { return __hiloint2double(perm(__double2hiint(d)), perm(__double2loint(d))); };
    v += moved(v, [](int x) { return __builtin_amdgcn_update_dpp(0, x, 0xb1, 0xf, 0xf, true); });
    v += moved(v, [](int x) { return __builtin_amdgcn_update_dpp(0, x, 0x4e, 0xf, 0xf, true); });
    v += moved(v, [](int x) { return __builtin_amdgcn_update_dpp(0, x, 0x141, 0xf, 0xf, true); });
    v += moved(v, [](int x) { return __builtin_amdgcn_update_dpp(0, x, 0x140, 0xf, 0xf, true); });
    {
        const u2_t hi = __builtin_amdgcn_permlane16_swap((uint32_t)__double2hiint(v), (uint32_t)__double2hiint(v), false, false);
        const u2_t lo = __builtin_amdgcn_permlane16_swap((uint32_t)__double2loint(v), (uint32_t)__double2loint(v), false, false);
        v = __hiloint2double((int)hi.x, (int)lo.x) + __hiloint2double((int)hi.y, (int)lo.y);
    }
    {
        const u2_t hi = __builtin_amdgcn_permlane32_swap((uint32_t)__double2hiint(v), (uint32_t)__double2hiint(v), false, false);
        const u2_t lo = __builtin_amdgcn_permlane32_swap((uint32_t)__double2loint(v), (uint32_t)__double2loint(v), false, false);
        v = __hiloint2double((int)hi.x, (int)lo.x) + __hiloint2double((int)hi.y, (int)lo.y);
    }
    return v;
}

// What the attention kernel needs to finish the projections itself: the raw output of the QKV matmul
// ([q heads | k heads | v heads], head_dim each), the optional per-head RMSNorm weights, the rotation, and the caches
// whose row `position` it writes.
struct AttnFront {
    const float* qkv;
    const float* q_norm_w;
    const float* k_norm_w;
    float eps, theta_scale, freq_scale;
    int neox;
    int num_heads, num_kv_heads;
    float* k_cache;
    float* v_cache;
};

// x of the lane whose number differs in bit B (and, for the mirrors, in the lower ones) inside a row of 16 lanes
template <int B>
__device__ __forceinline__ float other16(float x)
{
    constexpr int kCtrl = B == 0 ? 0xb1 : B == 1 ? 0x4e : B == 2 ? 0x141 : 0x140;    // quad_perm [1,0,3,2], [2,3,0,1], mirrors of 8 and 16
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kCtrl, 0xf, 0xf, true));
}
// x of lane L of the row of 16, in all its lanes
template <int L>
__device__ __forceinline__ float bcast16(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x150 + L, 0xf, 0xf, true));    // row_newbcast
}
typedef uint32_t lane_pair_t __attribute__((ext_vector_type(2)));
// one step of a sum over the four 16-lane rows of a wavefront that leaves a different value behind in each: rows 0 | 1 and 2 | 3
// (the halves of the wavefront) get a and b
__device__ __forceinline__ float rows_sum16(float a, float b)
{
    const lane_pair_t r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r.x) + __uint_as_float(r.y);
}
__device__ __forceinline__ float rows_sum32(float a, float b)
{
    const lane_pair_t r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r.x) + __uint_as_float(r.y);
}
__device__ __forceinline__ float rows_max(float x)
{
    lane_pair_t r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(r.x), __uint_as_float(r.y));
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r.x), __uint_as_float(r.y));
}

constexpr int log2_of(int n) { return n <= 1 ? 0 : 1 + log2_of(n / 2); }

// Sums over the 16 lanes of a row, NV of them at once, that leave value i only in the lanes that go on with it: at the step
// of lane bit B a lane keeps the half of the values that its bit names and hands the other half to its neighbour.  Value i
// ends in the lanes lane / 2^(4 - log2 NV) == i (NV = 32: values 2 lane and 2 lane + 1).  Sixteen sums cost 45 instructions
// instead of 64, and what follows (maximum, exponential, sum) runs once per value instead of once per value and lane.
template <int B, int NV>
__device__ __forceinline__ void scatter_sums(float (&v)[NV], int lane, int count)
{
    if constexpr (B >= 0) {
        if (count > 1) {
            const bool up = (lane >> B) & 1;
#pragma unroll
            for (int i = 0; i < count / 2; ++i) {
                const float keep = up ? v[i + count / 2] : v[i], give = up ? v[i] : v[i + count / 2];
                v[i] = keep + other16<B>(give);
            }
            scatter_sums<B - 1, NV>(v, lane, count / 2);
        } else {
            v[0] += other16<B>(v[0]);
            scatter_sums<B - 1, NV>(v, lane, 1);
        }
    }
}

template <int L, int N>
__device__ __forceinline__ float bcast_step(float x, int l)
{
    if constexpr (L + 1 < N) return l == L ? bcast16<L>(x) : bcast_step<L + 1, N>(x, l);
    else return bcast16<L>(x);
}
// x of lane l of the row of 16; l is a constant once the loops around are unrolled
__device__ __forceinline__ float bcast16_at(float x, int l) { return bcast_step<0, 16>(x, l); }

// grid (num_kv_heads, splits, q-head chunks): one workgroup serves G query heads that share a KV head, so every K / V
// row is loaded once for all of them.  8 wavefronts x 4 groups of 16 lanes; a group takes positions g, g + 32, ... of the
// split, U of them, all requested before the first is used (a split is 32 U positions, there is no second trip), lane l of a
// group holds the head dimensions l, l + 16, ... (PER of them).  The scores of a group's G x U (head, position) pairs are
// summed over its lanes by scatter_sums, so that every pair's exponential is evaluated in one lane (or in a few) and reaches
// the others by row_newbcast; a wavefront has one maximum per head, so that its groups' results add up without further factors;
// the wavefronts merge their softmax states in LDS.
// Bound: latency (launch, preparation of the heads, one trip to the caches), then HBM.  Against four wavefronts whose groups took
// the positions four at a time with one sum, exponential and running maximum per pair: 32 x 8 heads of 128 at 512 positions
// 6.6 -> 5.2 us, at 4001 positions (33 MB) 13.6 -> 10.6 us by the kernel trace; three Q8_0 layers and a head 182.1 -> 175.2.
// (K / V rows as 16-byte loads: the same on every shape.)
// Where a KV head has 3, 5, 6 or 7 query heads, a workgroup of the next power of two serves them all, the last one in the places
// that are left over (nothing of those is stored).
// Wavefronts per SIMD that the registers have to leave room for: two workgroups per CU for head dimensions of 192 (131 -> 128
// registers; 12 x 2 heads at 16000 and 32000 positions 102 -> 91 and 149 -> 132 us per two small layers).
template <int PER, int G>
constexpr int kAttnMinWaves = PER == 12 && G <= 4 ? 4 : 1;
template <int PER, int G, int U>
__global__ void __launch_bounds__(kAttnWaves * 64, (kAttnMinWaves<PER, G>)) attn_decode_kernel(float* k_cache, float* v_cache, const float* qkv, int group,
                                                                       int max_seq_len, int total, int split_len, float scale, int splits,
                                                                       int num_heads, float* __restrict__ partial, const AttnFront F,
                                                                       float* __restrict__ out_direct, const float* pre0, const float* pre1,
                                                                       int pre_floats)
{
    // (what the first loads need - the caches, the projections, the geometry - are leading scalar arguments: the hardware
    // delivers the first 14 dwords in SGPRs at wave launch, the rest is read from the argument block)
    constexpr int HD = 16 * PER;
    __shared__ float sm[kAttnWaves][G], sl[kAttnWaves][G], sacc[kAttnWaves][G][HD];
    __shared__ float sq[G][HD], sk[HD], sv[HD], tmp[kAttnWaves][HD];
    const int kvh = blockIdx.x, split = blockIdx.y;
    if (split == splits) {
        // One more row of workgroups than there are splits: they only read the vectors that the launches after this one
        // ask for first (the norm weights of the FFN and of the next layer) and leave.  Read from HBM by this kernel's
        // spare workgroups, the vectors wait in the memory-side cache (and, consecutive workgroups being dealt to
        // consecutive XCDs, in every L2) instead of queueing up behind a launch's first weight requests: 1.25 us per
        // RMSNorm launch, measured by leaving the vector out.
        if (blockIdx.z == 0) {
            for (int i = (int)threadIdx.x * 4; i < pre_floats; i += kAttnWaves * 64 * 4) {
                typedef float f4_t __attribute__((ext_vector_type(4)));
                // Ordinary loads with an empty use: the compiler owns their registers (written in asm, a load in flight could
                // land in registers that already hold the next address) and waits for them on every trip, two trips of
                // 2048 floats at a hidden size of 4096.  The trips hide behind the other workgroups' K / V rows: with all
                // eight requests of a thread in flight at once the launch took 6.5 instead of 6.35 us (32 heads, 60 and 200
                // positions, four runs each).
                f4_t a = {0.f, 0.f, 0.f, 0.f}, b = a;
                if (pre0) a = *reinterpret_cast<const f4_t*>(pre0 + i);
                if (pre1) b = *reinterpret_cast<const f4_t*>(pre1 + i);
                asm volatile("" ::"v"(a), "v"(b));
            }
        }
        return;
    }
    const int h0 = kvh * group + blockIdx.z * G;                     // first query head of this workgroup
    const int heads = min(G, group - (int)blockIdx.z * G);           // of its places, how many hold a head of their own
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lg = lane & 15, grp = (wave << 2) | (lane >> 4);
    const float* kb = k_cache + (int64_t)kvh * max_seq_len * HD;
    const float* vb = v_cache + (int64_t)kvh * max_seq_len * HD;
    const int position = total - 1;
    const bool last = split == splits - 1;                           // the split that holds the new position
    // U rows of K and of V per group, all requested before the first is used and ahead of the work on the projections below,
    // which does not depend on them
    const int t_end = min(total, (split + 1) * split_len);
    const int t0 = split * split_len + grp;
    float kr[U][PER], vr[U][PER];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int64_t row = (int64_t)min(t0 + kAttnGroups * u, t_end - 1) * HD + lg;      // rows past the split: a valid row, unused
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            kr[u][j] = kb[row + 16 * j];
            vr[u][j] = vb[row + 16 * j];
        }
    }

    // ---- the projections' last steps, per head: RMSNorm over the head (ggml_rms_norm, then * weight), RoPE at
    // `position` (ggml_rope_ext with n_dims = head_dim: ggml-cpu/ops.cpp:5549-5563, :5636-5652).  Every workgroup
    // prepares its own query heads; the workgroup of the last split also prepares the new key / value row, uses it
    // from LDS and (query-head chunk 0 only) writes it to the caches.
    {
        constexpr int kPer = (HD + 63) / 64, kPairs = (HD / 2 + 63) / 64;
        constexpr int half = HD / 2;
        const int nprep = G + (last ? 1 : 0);
        auto head_src = [&](int hh) { return qkv + (int64_t)(hh < G ? h0 + min(hh, heads - 1) : num_heads + kvh) * HD; };
        // the wavefront's first head is requested before the angles are worked out
        float xv[kPer];
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int d = lane + 64 * j;
            xv[j] = (wave < nprep && d < HD) ? head_src(wave)[d] : 0.f;
        }
        float cs[kPairs], sn[kPairs];
        {
            // the reference builds theta by repeated multiplication; the same float products in the same order.  One
            // uniform chain of half - 1 products, every lane keeping the value of its own pair (a loop of lane-dependent
            // length costs several times as many instructions per product).
            // theta_i = theta_(i-1) * theta_scale, i = lane + 64 j: every step each lane takes its lower neighbour's value
            // times theta_scale (lane 0: its own value times one), so that after 63 steps lane i has been through exactly
            // the products 1 .. i of the chain - one instruction per step instead of a multiply, a compare and a select.
            const float factor = lane == 0 ? 1.0f : F.theta_scale;
            float chain = (float)position;
#pragma unroll
            for (int j = 0; j < kPairs; ++j) {
                if (j > 0) chain = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(chain), 63)) * F.theta_scale;
                const int steps = min(half - 64 * j, 64) - 1;
                for (int i = 0; i < steps; ++i) {
                    const int below = __builtin_amdgcn_update_dpp(__float_as_int(chain), __float_as_int(chain), 0x138, 0xf, 0xf, false);   // wave_shr:1
                    chain = __int_as_float(below) * factor;
                }
                cs[j] = chain;
            }
#pragma unroll
            for (int j = 0; j < kPairs; ++j) {
                const float ang = F.freq_scale * cs[j];
                sincosf(ang, &sn[j], &cs[j]);
            }
        }
        for (int hh = wave; hh < nprep; hh += kAttnWaves) {          // uniform per wavefront
            const bool is_q = hh < G;
            const float* src = head_src(hh);
            const float* nw = is_q ? F.q_norm_w : F.k_norm_w;
            if (hh != wave) {
#pragma unroll
                for (int j = 0; j < kPer; ++j) {
                    const int d = lane + 64 * j;
                    xv[j] = d < HD ? src[d] : 0.f;
                }
            }
            float rs = 1.f;
            if (nw) {
                // ggml-cpu/ops.cpp:3646-3695: sum of squares in double, scale = 1 / sqrtf(mean + eps)
                double ss = 0.0;
#pragma unroll
                for (int j = 0; j < kPer; ++j) ss += (double)(xv[j] * xv[j]);
                ss = wave_sum(ss);
                rs = 1.0f / sqrtf((float)(ss / (double)HD) + F.eps);
            }
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                const int d = lane + 64 * j;
                if (d < HD) tmp[wave][d] = nw ? (xv[j] * rs) * nw[d] : xv[j];
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // the wavefront's own LDS writes before its reads
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            float* dst = is_q ? sq[hh] : sk;
            const float by = is_q ? scale : 1.0f;
            float* cache = (!is_q && blockIdx.z == 0) ? k_cache + ((int64_t)kvh * max_seq_len + position) * HD : nullptr;
#pragma unroll
            for (int j = 0; j < kPairs; ++j) {
                const int p = lane + 64 * j;
                if (p < half) {
                    const int i0 = F.neox ? p : 2 * p, i1 = F.neox ? p + half : 2 * p + 1;
                    const float x0 = tmp[wave][i0], x1 = tmp[wave][i1];
                    const float r0 = x0 * cs[j] - x1 * sn[j], r1 = x0 * sn[j] + x1 * cs[j];
                    dst[i0] = r0 * by;
                    dst[i1] = r1 * by;
                    if (cache) {
                        cache[i0] = r0;
                        cache[i1] = r1;
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // tmp is reused by this wavefront's next head
            __builtin_amdgcn_wave_barrier();
        }
        if (last) {
            const float* src = qkv + (int64_t)(num_heads + F.num_kv_heads + kvh) * HD;
            float* cache = blockIdx.z == 0 ? v_cache + ((int64_t)kvh * max_seq_len + position) * HD : nullptr;
            for (int d = threadIdx.x; d < HD; d += kAttnWaves * 64) {
                const float v = src[d];
                sv[d] = v;
                if (cache) cache[d] = v;
            }
        }
        __syncthreads();
    }
    if (last) {       // uniform: the new position's row is not in the caches yet (another workgroup may be writing it)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // Slots past the split hold a clamped row (the row being written by this very launch, or whatever the cache memory
            // held): their values must not reach the sums, not even multiplied by a zero weight (0 * NaN), so they are
            // replaced, not scaled (the scores below).
            const int t = t0 + kAttnGroups * u;
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                kr[u][j] = t == position ? sk[lg + 16 * j] : kr[u][j];
                vr[u][j] = t == position ? sv[lg + 16 * j] : t < t_end ? vr[u][j] : 0.f;
            }
        }
    }
    // scores: value g U + u is head g, position u of the group
    constexpr int NV = G * U;
    constexpr int kPerLane = NV > 16 ? NV / 16 : 1;                  // values a lane ends with
    constexpr int kShift = NV > 16 ? 0 : 4 - log2_of(NV);            // lane >> kShift: the (first) value of a lane, / kPerLane
    constexpr int kUInLane = kPerLane;                               // positions of a head that share a lane
    constexpr int kULanes = log2_of(U / kUInLane);                   // lane bits kShift .. that number a head's positions
    float sc[NV];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        float qr[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) qr[j] = sq[g][lg + 16 * j];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float d = 0.f;
#pragma unroll
            for (int j = 0; j < PER; ++j) d += qr[j] * kr[u][j];
            sc[g * U + u] = d;
        }
    }
    scatter_sums<3, NV>(sc, lg, NV);
    if (last) {
#pragma unroll
        for (int r = 0; r < kPerLane; ++r) {
            const int u = ((lg >> kShift) * kPerLane + r) & (U - 1);
            if (t0 + kAttnGroups * u >= t_end) sc[r] = -INFINITY;
        }
    }
    auto over_positions = [&](float x, auto op) {                    // of the lane's head, inside the group
        if constexpr (kULanes > 0) x = op(x, other16<kShift>(x));
        if constexpr (kULanes > 1) x = op(x, other16<kShift + 1>(x));
        return x;
    };
    float m = sc[0];
#pragma unroll
    for (int r = 1; r < kPerLane; ++r) m = fmaxf(m, sc[r]);
    m = rows_max(over_positions(m, [](float a, float b) { return fmaxf(a, b); }));
    const float mref = m == -INFINITY ? 0.f : m;                     // a wavefront without a live position: weights of zero
    float l = 0.f;
#pragma unroll
    for (int r = 0; r < kPerLane; ++r) {
        sc[r] = expf(sc[r] - mref);
        l += sc[r];
    }
    l = over_positions(l, [](float a, float b) { return a + b; });
    l = rows_sum16(l, l);
    l = rows_sum32(l, l);
    // the lane that holds value i (NV = 32: two values per lane)
    auto lane_of = [&](int i) { return (i / kPerLane) << kShift; };
    if (lane < 16 && (lane & ((1 << (kShift + kULanes)) - 1)) == 0) {
        const int g = lane >> (kShift + kULanes);
        if (g < G) {
            sm[wave][g] = m;
            sl[wave][g] = l;
        }
    }
    constexpr int NF = (G * PER + 3) / 4 * 4;
    float acc[NF];
#pragma unroll
    for (int f = G * PER; f < NF; ++f) acc[f] = 0.f;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        float pw[U];
#pragma unroll
        for (int u = 0; u < U; ++u) pw[u] = bcast16_at(sc[(g * U + u) % kPerLane], lane_of(g * U + u));
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            float a = 0.f;
#pragma unroll
            for (int u = 0; u < U; ++u) a += pw[u] * vr[u][j];
            acc[g * PER + j] = a;
        }
    }
    // the four groups of the wavefront: row r of it ends with the sums of acc[4 q + r]
    float* const my_acc = &sacc[wave][0][0];
#pragma unroll
    for (int q = 0; q < NF / 4; ++q) {
        const float t = rows_sum32(rows_sum16(acc[4 * q], acc[4 * q + 1]), rows_sum16(acc[4 * q + 2], acc[4 * q + 3]));
        const int f = 4 * q + (lane >> 4), g = f / PER, j = f - g * PER;
        if (G * PER % 4 == 0 || f < G * PER) my_acc[g * HD + lg + 16 * j] = t;
    }
    __syncthreads();
    // the wavefronts: thread (g, d) of the first heads * HD threads
    for (int i = threadIdx.x; i < heads * HD; i += kAttnWaves * 64) {
        const int g = i / HD, d = i - g * HD;
        float mm = -INFINITY;
#pragma unroll
        for (int w = 0; w < kAttnWaves; ++w) mm = fmaxf(mm, sm[w][g]);
        float ll = 0.f, out = 0.f;
#pragma unroll
        for (int w = 0; w < kAttnWaves; ++w) {
            const float f = sm[w][g] == -INFINITY ? 0.f : expf(sm[w][g] - mm);
            ll += sl[w][g] * f;
            out += sacc[w][g][d] * f;
        }
        if (out_direct) {
            out_direct[(int64_t)(h0 + g) * HD + d] = out / ll;       // a single split: this is the result
            continue;
        }
        float* dst = partial + ((int64_t)(h0 + g) * splits + split) * (kMaxHeadDim + 2);
        if (d == 0) {
            dst[0] = mm;
            dst[1] = ll;
        }
        dst[2 + d] = out;
    }
}

// one workgroup per head: wavefront w merges splits w, w + WAVES, ... (four rows in flight), the wavefronts meet in LDS
template <int WAVES>
__global__ void __launch_bounds__(WAVES * 64) attn_combine_kernel(const float* __restrict__ partial, int splits, int head_dim,
                                                                        float* __restrict__ out)
{
    constexpr int kPer = kMaxHeadDim / 64, kRow = kMaxHeadDim + 2;
    __shared__ float sacc[WAVES][kMaxHeadDim], sl[WAVES];
    const int h = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float* base = partial + (int64_t)h * splits * kRow;
    float ms[4], ls[4], v[4][kPer];
    auto load_rows = [&](int s0) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int s = s0 + u * WAVES;
            const bool live = s < splits;
            const float* p = base + (int64_t)(live ? s : s0) * kRow;
            ms[u] = live ? p[0] : -INFINITY;
            ls[u] = live ? p[1] : 0.f;
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                const int d = lane + 64 * j;
                v[u][j] = (live && d < head_dim) ? p[2 + d] : 0.f;
            }
        }
    };
    // When one batch of rows per wavefront covers the splits (16 of four wavefronts, 64 of sixteen), it is requested before
    // the maximum over all splits is worked out (every wavefront computes it: independent loads, one pass), so that the two
    // round trips overlap: 0.35 us per layer.  (With more batches the early request measured 0.3 us slower.)
    constexpr int kBatch = 4 * WAVES;
    const bool early = splits <= kBatch;
    if (early && wave < splits) load_rows(wave);
    float mm = -INFINITY;
    for (int s = lane; s < splits; s += 64) mm = fmaxf(mm, base[(int64_t)s * kRow]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mm = fmaxf(mm, __shfl_xor(mm, o));
    float acc[kPer], ll = 0.f;
#pragma unroll
    for (int j = 0; j < kPer; ++j) acc[j] = 0.f;
    for (int s0 = wave; s0 < splits; s0 += kBatch) {
        if (!early) load_rows(s0);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const float f = ms[u] == -INFINITY ? 0.f : expf(ms[u] - mm);
            ll += ls[u] * f;
#pragma unroll
            for (int j = 0; j < kPer; ++j) acc[j] += v[u][j] * f;
        }
    }
    if (lane == 0) sl[wave] = ll;
#pragma unroll
    for (int j = 0; j < kPer; ++j) sacc[wave][lane + 64 * j] = acc[j];
    __syncthreads();
    if (wave == 0) {
        float lt = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) lt += sl[w];
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int d = lane + 64 * j;
            float a = 0.f;
#pragma unroll
            for (int w = 0; w < WAVES; ++w) a += sacc[w][d];
            if (d < head_dim) out[(int64_t)h * head_dim + d] = a / lt;
        }
    }
}

}  // namespace

// (at least what any shorter context takes, so that a workspace that served one position serves the next)
size_t attention_decode_ws_bytes(int num_heads, int total)
{
    const int splits = std::max((total + 4 * kAttnGroups - 1) / (4 * kAttnGroups), kFewSplits);
    return (size_t)num_heads * splits * (kMaxHeadDim + 2) * sizeof(float);
}

bool launch_attention_decode(const float* qkv, const float* q_norm_w, const float* k_norm_w, float eps, float rope_base,
                             float rope_freq_scale, int rope_mode, float* k_cache, float* v_cache, int num_heads, int num_kv_heads,
                             int head_dim, int max_seq_len, int position, float* partial_ws, float* out, hipStream_t stream,
                             const float* prefetch0, const float* prefetch1, int prefetch_floats)
{
    const int total = position + 1;
    if (num_kv_heads <= 0 || num_heads % num_kv_heads != 0 || total <= 0 || total > max_seq_len) {
        set_last_error("layer decode: bad head counts or position.");
        return false;
    }
    if (rope_mode != 0 && rope_mode != 2) {
        set_last_error("layer decode: rope mode must be 0 (adjacent pairs) or 2 (NeoX halves).");
        return false;
    }
    AttnFront front{};
    front.qkv = qkv;
    front.q_norm_w = q_norm_w;
    front.k_norm_w = k_norm_w;
    front.eps = eps;
    front.theta_scale = powf(rope_base, -2.0f / (float)head_dim);           // ggml-cpu/ops.cpp:5711
    front.freq_scale = rope_freq_scale;
    front.neox = rope_mode == 2 ? 1 : 0;
    front.num_heads = num_heads;
    front.num_kv_heads = num_kv_heads;
    front.k_cache = k_cache;
    front.v_cache = v_cache;
    const int rows = attn_rows(num_heads, num_kv_heads, total), split_len = kAttnGroups * rows;
    const int splits = (total + split_len - 1) / split_len;
    if (splits > 65535) {
        set_last_error("layer decode: context too long for one launch.");
        return false;
    }
    const float scale = 1.0f / sqrtf((float)head_dim);
    const int group = num_heads / num_kv_heads;
    // query heads per workgroup: as many as share the KV head (its rows are then loaded once), fewer while that leaves
    // the launch with too few workgroups to hide its latency (64 or 256 as the line: 1 to 22 % longer at the contexts between, per
    // two small layers: 8 x 1 heads of 256 at 6000 positions 57 / 61 / 58 us with 128 / 64 / 256, at 12000 71 / 75 / 84)
    int g = group % 8 == 0 ? 8 : group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
    while (g > 2 && num_kv_heads * splits * (group / g) < 128) g >>= 1;
    // Groups of 3, 5, 6 and 7 heads in one workgroup with places left over, once that makes 184 workgroups; with one or two
    // heads each, every row was loaded two to seven times, and a workgroup of eight wavefronts took up to 8 % longer for it than
    // the four of a former build.  us per two small layers, g of the rule above / all heads: 40 x 8 heads of 128 at 1500 positions (192
    // workgroups) 53.8 / 53.9, 2047 59.8 / 55.8, 6000 101.8 / 75.6, 16000 232 / 106, 28 x 4 at 8191 107 / 62, 24 x 8 at 4000
    // 61.9 / 55.6, 28 x 4 of 64 at 3000 (188) 49.2 / 45.9, 24 x 4 of 256 69.2 / 68.2; short of the line 40 x 8 at 1023 (136) 49.4 / 51.4, 24 x 4 of 256 at 2048 (132) 59 / 66.
    constexpr int kEnough = 184;
    if (group < 8 && (group & (group - 1)) != 0 && num_kv_heads * splits >= kEnough) g = group == 3 ? 4 : 8;
    // (vectors to prefetch: whole float4s at 16-byte aligned addresses, else none)
    const bool pre = (prefetch0 || prefetch1) && prefetch_floats > 0 && prefetch_floats % 4 == 0 && splits < 65535 &&
                     ((reinterpret_cast<uintptr_t>(prefetch0) | reinterpret_cast<uintptr_t>(prefetch1)) & 15) == 0;
    const dim3 grid(num_kv_heads, splits + (pre ? 1 : 0), (group + g - 1) / g), block(kAttnWaves * 64);
#define TSHIP_ATTN_LAUNCH_U(PER, GG, U)                                                                                         \
    hipLaunchKernelGGL((attn_decode_kernel<PER, GG, U>), grid, block, 0, stream, front.k_cache, front.v_cache, front.qkv, group,     \
                       max_seq_len, total, split_len, scale, splits, num_heads, partial_ws, front, splits == 1 ? out : nullptr,           \
                       pre ? prefetch0 : nullptr, pre ? prefetch1 : nullptr, pre ? prefetch_floats : 0)
#define TSHIP_ATTN_LAUNCH(PER, GG)                                           \
    if (rows == 2)          TSHIP_ATTN_LAUNCH_U(PER, GG, 2);              \
    else TSHIP_ATTN_LAUNCH_U(PER, GG, 4)
#define TSHIP_ATTN_G(PER)                                                    \
    switch (g) {                                                             \
    case 8: TSHIP_ATTN_LAUNCH(PER, 8); break;                                \
    case 4: TSHIP_ATTN_LAUNCH(PER, 4); break;                                \
    case 2: TSHIP_ATTN_LAUNCH(PER, 2); break;                                \
    default: TSHIP_ATTN_LAUNCH(PER, 1); break;                               \
    }
    switch (head_dim) {
    case 64: TSHIP_ATTN_G(4) break;
    case 80: TSHIP_ATTN_G(5) break;
    case 96: TSHIP_ATTN_G(6) break;
    case 128: TSHIP_ATTN_G(8) break;
    case 192: TSHIP_ATTN_G(12) break;
    case 256: TSHIP_ATTN_G(16) break;
    default: set_last_error("layer decode: head_dim must be one of 64, 80, 96, 128, 192, 256."); return false;
    }
#undef TSHIP_ATTN_G
#undef TSHIP_ATTN_LAUNCH
#undef TSHIP_ATTN_LAUNCH_U
    if (!hip_ok(hipGetLastError(), "attention launch")) return false;
    if (splits == 1) return true;
    // Four wavefronts request up to 16 splits' rows in one round trip; more splits take sixteen, which cover 64, instead of
    // further dependent trips (32 splits, 32 heads: three layers at 4001 positions 196.5 -> 194.8 us; four layers of 32 heads
    // at 8192 / 16000 / 30000 positions 190 -> 180, 263 -> 243, 404 -> 364 us).
    if (splits <= 16)
        hipLaunchKernelGGL(attn_combine_kernel<4>, dim3(num_heads), dim3(4 * 64), 0, stream, partial_ws, splits, head_dim, out);
    else
        hipLaunchKernelGGL(attn_combine_kernel<16>, dim3(num_heads), dim3(16 * 64), 0, stream, partial_ws, splits, head_dim, out);
    return hip_ok(hipGetLastError(), "attention combine launch");
}

}  // namespace tship
