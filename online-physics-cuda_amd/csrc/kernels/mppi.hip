// A world model's MPPI planner on gfx950: rollouts of a learned ODE on the matrix cores and the softmin plan update.
//
// The reference plans with one thread a future, the dynamics MLP evaluated in fp32 registers with the weights in shared
// memory (src/field/mind/WorldModel.cpp:192-240). Here a wave carries 16 or 32 futures through the whole horizon without
// leaving its registers: a layer is W (A: 16 outputs x 16 inputs a product, fp16, two products a fragment from LDS) times the
// futures' inputs (B: 16 inputs x 16 futures) summed in fp32 from 0, a block of 16 inputs after the other, and the bias; a
// product's D (lane l: future l % 16, outputs 4 (l / 16)..+3 of a block of 16) is, after tanh and rounding to fp16, the next
// layer's B with no exchange between lanes. The states stay in D's layout in fp32; the last layer's rates move them there.
// The update weighs every future by exp(-(J - J_min) / lambda) and sums the futures one by one. Every sum's order is fixed
// (a layer's inputs in blocks of 16, a cost's features four apart, the futures in turn), whatever the number of agents,
// futures and tiles a wave: the same inputs give the same plan, bit for bit, and tests/golden/mppi/plans.npz holds some.
#include "fe_mppi.h"
#include "fe_hip.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <stdexcept>
#include <string>
#include <vector>

namespace {

typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef unsigned long long u64;

constexpr int kMaxWidth = 128; // hidden width
constexpr int kMaxState = 64;  // inputs: features and the two actions

struct Desc {
    int F, fb, horizon, samples; // fb: blocks of 16 features
    const half8* frags;    // the weights' fragments: layer 1, 2, 3, each [output block][32 inputs][lane]
    const float4v* tables; // b1, b2 [hidden], b3 [16 fb], shift, inscale [32 NC], scale, target, weight [16 fb]
    float action_weight;
};

// The input that element e of lane group g holds of the 32 of fragment c: two blocks of a product's D side by side.
__host__ __device__ inline int kfeat(int c, int g, int e) { return 32 * c + 16 * (e >> 2) + 4 * g + (e & 3); }

// The noise of (agent id, tick, future, step, axis): a standard normal by Box-Muller from two uniforms, each the top 24
// bits of a 64-bit mix (splitmix64's finaliser, Steele, Lea and Flood 2014) of the key and of the key's mix.
__host__ __device__ inline u64 mix64(u64 h)
{
    h ^= h >> 30;
    h *= 0xbf58476d1ce4e5b9ull;
    h ^= h >> 27;
    h *= 0x94d049bb133111ebull;
    h ^= h >> 31;
    return h;
}
// The part of a key that is the same for every future and step of one agent's plan; the key of (future k, step t,
// axis d) is noise_base ^ (k << 24) ^ (t << 8) ^ d.
__host__ __device__ inline u64 noise_base(u64 id, u64 tick)
{
    return mix64(id * 0x9e3779b97f4a7c15ull + 1) ^ mix64(tick * 0xd1b54a32d192ed03ull + 2);
}
// The hardware's logarithm, square root and cosine (v_log_f32, v_sqrt_f32, v_cos_f32, the last taking turns, so
// cos(2 pi u2) is one instruction): a few ulp, where the library's range reductions were a large share of a step.
__device__ inline float gauss(u64 key)
{
    const u64 a = mix64(key), b = mix64(a ^ 0x632be59bd9b4e019ull);
    const float u1 = ((float)(a >> 40) + 0.5f) * (1.0f / 16777216.0f);
    const float u2 = ((float)(b >> 40) + 0.5f) * (1.0f / 16777216.0f);
    return __builtin_amdgcn_sqrtf(-2.0f * 0.6931471805599453f * __builtin_amdgcn_logf(u1)) * __builtin_amdgcn_cosf(u2);
}

// tanh u = 1 - 2 / (1 + e^(2u)) through the hardware exponential and reciprocal: a few ulp of fp32, below the fp16
// rounding of the activation it becomes; the library tanhf's long polynomial sequence was most of a layer's issue slots.
// Saturates to +-1 (e^(2u) overflowing to inf, or to 0). Not a fused multiply-add: with the rounding to fp16 behind it the
// compiler takes one instruction that rounds once, and the activation's last bit changes.
__device__ __forceinline__ float fast_tanh(float u)
{
    const float e = __builtin_amdgcn_exp2f((2.0f * 1.4426950408889634f) * u); // e^(2u), 2 log2(e) folded
    return 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + e);
}

// A layer's bias and tanh, rounded into the next layer's inputs (zero past the hidden units).
template <int HB, int Q>
__device__ __forceinline__ void activate(float4v (&z)[HB][Q], const float4v* b, int g, half8 (&h)[Q][(HB + 1) / 2])
{
#pragma unroll
    for (int ob = 0; ob < HB; ++ob) {
        const float4v bias = b[4 * ob + g];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            z[ob][q] += bias;
        }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
#pragma unroll
        for (int c = 0; c < (HB + 1) / 2; ++c) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int ob = 2 * c + (e >> 2);
                h[q][c][e] = ob < HB ? (_Float16)fast_tanh(z[ob < HB ? ob : 0][q][e & 3]) : (_Float16)0.0f;
            }
        }
    }
}

// Fragments and tables (float4) of a net with HB blocks of 16 hidden units, NC fragments of inputs and fb blocks of features.
__host__ __device__ constexpr int frag_count(int HB, int NC, int fb) { return HB * NC + (HB + fb) * ((HB + 1) / 2); }
__host__ __device__ constexpr int table_count(int HB, int NC, int fb) { return 4 * (2 * HB + 4 * NC + 4 * fb); }
constexpr int lds_bytes(int HB, int NC, int fb) { return frag_count(HB, NC, fb) * 1024 + table_count(HB, NC, fb) * 16; }

// A fragment's 32 inputs for all Q tiles as two products of 16, the first block and (`both`) the second: the one deep product
// adds them in an order of its own, which moves activations across fp16 boundaries. A block of zeros changes nothing.
template <int Q, typename In>
__device__ __forceinline__ void mfma(half8 w, const In& in, float4v (&acc)[Q], bool both)
{
    const half4 w0 = __builtin_shufflevector(w, w, 0, 1, 2, 3), w1 = __builtin_shufflevector(w, w, 4, 5, 6, 7);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        acc[q] = __builtin_amdgcn_mfma_f32_16x16x16f16(w0, __builtin_shufflevector(in(q), in(q), 0, 1, 2, 3), acc[q], 0, 0, 0);
    }
    if (both) {
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            acc[q] = __builtin_amdgcn_mfma_f32_16x16x16f16(w1, __builtin_shufflevector(in(q), in(q), 4, 5, 6, 7), acc[q], 0, 0, 0);
        }
    }
}

// Lane group g's four values for features 4g..4g + 3 of a block to those of features g, g + 4, g + 8, g + 12 (a 4 x 4
// transpose over the wave's four groups of 16 lanes): v_permlane32_swap exchanges a register's upper 32 lanes with another's
// lower ones, v_permlane16_swap its odd rows of 16 with another's even ones.
__device__ __forceinline__ void swap32(float& a, float& b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap16(float& a, float& b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void by_fours(float (&v)[4])
{
    swap32(v[0], v[2]);
    swap32(v[1], v[3]);
    swap16(v[0], v[1]);
    swap16(v[2], v[3]);
}

// A wave takes 16 Q futures of an agent at a time; wave w of the grid the items w, w + waves, ... (agent-major). Actions into
// acts[agent][t][k][axis], each future's cost into cost[agent][k]. The noise is drawn by every lane: with two tiles (Q = 2)
// lane l the future l / 2, axis l % 2 of the step; with one, the lanes 32.. draw the step after. The weights and the tables
// are read from LDS where they are used (two tiles to a read).
// Bound by the hidden units' tanh, two quarter-rate instructions each: about 165 us of 256 agents x 512 futures x 32 steps with
// 16 features and 64 hidden units, which take 229 (784 when each layer's activations went through LDS and its weights were
// read from memory a tile at a time). Products of 32 inputs that start from the bias would take 210, and give other bits.
template <int HB, int NC, int Q>
__global__ __launch_bounds__(256) void k_mppi_rollout(Desc d, const float* __restrict__ obs, const float* __restrict__ mean,
    const unsigned* __restrict__ ids, float* __restrict__ acts, float* __restrict__ cost, u64 tick, float sigma, float dt, unsigned items,
    unsigned per_agent)
{
    constexpr int HC = (HB + 1) / 2;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    half8* W1 = reinterpret_cast<half8*>(lds);
    const half8* W2 = W1 + HB * NC * 64;
    const half8* W3 = W2 + HB * HC * 64;
    const int fb = d.fb, frags = frag_count(HB, NC, fb) * 64, tables = table_count(HB, NC, fb);
    float4v* b1 = reinterpret_cast<float4v*>(W1 + frags);
    const float4v *b2 = b1 + 4 * HB, *b3 = b2 + 4 * HB, *shift = b3 + 4 * fb, *inscale = shift + 8 * NC, *scale = inscale + 8 * NC,
                  *target = scale + 4 * fb, *weight = target + 4 * fb;
    for (int i = (int)threadIdx.x; i < frags; i += 256) {
        W1[i] = d.frags[i];
    }
    for (int i = (int)threadIdx.x; i < tables; i += 256) {
        b1[i] = d.tables[i];
    }
    __syncthreads();
    const int l = (int)(threadIdx.x & 63u), n = l & 15, g = l >> 4;
    const int F = d.F, H = d.horizon, K = d.samples;
    const unsigned wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4u + (threadIdx.x >> 6)));
    for (unsigned item = wave; item < items; item += gridDim.x * 4u) {
        const long long agent = (long long)(item / per_agent);
        const int k0 = (int)(item % per_agent) * 16 * Q;
        const u64 base = noise_base(ids[agent], tick);
        float4v st[Q][2 * NC];
#pragma unroll
        for (int b = 0; b < 2 * NC; ++b) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int f = 16 * b + 4 * g + r;
                const float x = f < F ? obs[agent * F + f] : 0.0f;
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    st[q][b][r] = x;
                }
            }
        }
        float J[Q] = {}, drawn = 0.0f;
        for (int t = 0; t < H; ++t) {
            asm volatile("" ::: "memory"); // what LDS holds is read again each step: kept in registers it would spill
            if (Q == 2 || (t & 1) == 0) {
                const int row = Q == 2 ? l >> 1 : (l >> 1) & 15, axis = l & 1, step = Q == 2 ? t : t + (l >> 5), k = k0 + row;
                if (step < H) {
                    const float e = k == 0 ? 0.0f : gauss(base ^ ((u64)k << 24) ^ ((u64)step << 8) ^ (u64)axis);
                    drawn = fminf(fmaxf(mean[(agent * H + step) * 2 + axis] + sigma * e, -1.0f), 1.0f);
                    if (k < K) {
                        acts[((agent * H + step) * K + k) * 2 + axis] = drawn;
                    }
                }
            }
            float ax[Q], ay[Q];
            half8 in[Q][NC];
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const int from = 2 * (16 * q + n) + (Q == 2 ? 0 : 32 * (t & 1));
                ax[q] = __shfl(drawn, from);
                ay[q] = __shfl(drawn, from + 1);
            }
            // the inputs (state, then action), normalised, in fp16; zero past them
#pragma unroll
            for (int b = 0; b < 2 * NC; ++b) {
                const float4v sh = shift[4 * b + g], sc = inscale[4 * b + g];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int f = 16 * b + 4 * g + r;
#pragma unroll
                    for (int q = 0; q < Q; ++q) {
                        const float x = f < F ? st[q][b][r] : (f == F ? ax[q] : (f == F + 1 ? ay[q] : 0.0f));
                        in[q][b >> 1][4 * (b & 1) + r] = (_Float16)((x - sh[r]) * sc[r]);
                    }
                }
            }
            half8 h[Q][HC];
            float4v z[HB][Q];
#pragma unroll
            for (int ob = 0; ob < HB; ++ob) {
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    z[ob][q] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
                }
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    mfma(W1[(ob * NC + c) * 64 + l], [&](int q) { return in[q][c]; }, z[ob], true);
                }
            }
            activate<HB, Q>(z, b1, g, h);
            asm volatile("" ::: "memory");
#pragma unroll
            for (int ob = 0; ob < HB; ++ob) {
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    z[ob][q] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
                }
#pragma unroll
                for (int c = 0; c < HC; ++c) {
                    mfma(W2[(ob * HC + c) * 64 + l], [&](int q) { return h[q][c]; }, z[ob], 2 * c + 1 < HB);
                }
            }
            activate<HB, Q>(z, b2, g, h);
            asm volatile("" ::: "memory");
            // the rates, the states they move, and the states' part of the step's cost
            float c[Q] = {};
#pragma unroll
            for (int b = 0; b < 2 * NC; ++b) {
                if (b < fb) {
                    const float4v bias = b3[4 * b + g], sc = scale[4 * b + g], to = target[4 * b + g], wt = weight[4 * b + g];
                    float4v v[Q];
#pragma unroll
                    for (int q = 0; q < Q; ++q) {
                        v[q] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
                    }
#pragma unroll
                    for (int k = 0; k < HC; ++k) {
                        mfma(W3[(b * HC + k) * 64 + l], [&](int q) { return h[q][k]; }, v, 2 * k + 1 < HB);
                    }
#pragma unroll
                    for (int q = 0; q < Q; ++q) {
                        v[q] += bias;
                        float term[4];
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            st[q][b][r] += dt * v[q][r] * sc[r];
                            const float e = st[q][b][r] - to[r];
                            term[r] = wt[r] * e * e;
                        }
                        by_fours(term);
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            c[q] += term[r];
                        }
                    }
                }
            }
            // the four lane groups' features (four apart each) added in a fixed order
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                c[q] += __shfl_xor(c[q], 16);
                c[q] += __shfl_xor(c[q], 32);
                J[q] += c[q] + d.action_weight * (ax[q] * ax[q] + ay[q] * ay[q]);
            }
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int k = k0 + 16 * q + n;
            if (g == 0 && k < K) {
                cost[agent * K + k] = J[q];
            }
        }
    }
}

// The new plan: the futures' actions weighted by exp(-(J - J_min) / lambda), lambda a quarter of (mean cost - least cost), at
// least 1e-4. A block an agent: the least cost, the costs' sum and each future's weight once (in LDS), then a lane a (step,
// axis) of the first waves, the futures added in their order: a chain of K adds, which reads LDS. All threads bring the next
// run of futures there, its loads in flight beside the chain: 13 us for 256 agents x 512 futures x 32 steps, 4 x 32 futures
// 4 us (18-25 where a lane reads its own actions from memory, eight or 256 of them in flight; 8 as a tree over the lanes, whose
// sums are others).
constexpr int kMaxSamples = 1024;
constexpr int kUpdateThreads = 512;
constexpr int kRunFloats = 8192; // a run's actions: 128 futures up to 32 steps, 64 past them
__global__ __launch_bounds__(kUpdateThreads) void k_mppi_update(const float* __restrict__ cost, const float* __restrict__ acts,
    float* __restrict__ mean, int K, int H)
{
    constexpr int kPairs = kRunFloats / 2 / kUpdateThreads;
    __shared__ __attribute__((aligned(16))) float cs[kMaxSamples];
    __shared__ __attribute__((aligned(16))) float run[kRunFloats + 128]; // a step's futures a row, two floats of padding each
    __shared__ float lo_s, lam_s;
    const long long agent = (long long)blockIdx.x;
    const int q = (int)threadIdx.x;
    const int lt = H > 32 ? 6 : 7, T = 1 << lt, pitch = 2 * T + 2; // futures a run
    const float* a = acts + agent * H * 2 * K;
    // pair i of a run: future i % T of step i / T, both axes
    float2 held[kPairs];
    auto fetch = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kPairs; ++u) {
            const int i = q + u * kUpdateThreads, t = i >> lt, k = k0 + (i & (T - 1));
            held[u] = t < H && k < K ? *reinterpret_cast<const float2*>(a + (t * K + k) * 2) : make_float2(0.0f, 0.0f);
        }
    };
    auto put = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kPairs; ++u) {
            const int i = q + u * kUpdateThreads;
            *reinterpret_cast<float2*>(run + (i >> lt) * pitch + 2 * (i & (T - 1))) = held[u];
        }
    };
    fetch(0);
    for (int k = q; k < K; k += kUpdateThreads) {
        cs[k] = cost[agent * K + k];
    }
    put();
    __syncthreads();
    fetch(T);
    if (q < 64) {
        float lo = cs[0], sum = 0.0f;
        for (int k = q; k < K; k += 64) {
            lo = fminf(lo, cs[k]);
        }
        for (int m = 32; m > 0; m >>= 1) {
            lo = fminf(lo, __shfl_xor(lo, m));
        }
        for (int k = 0; k < K; k += 16) { // added in order, sixteen to a wait
            float4v c[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                c[i] = *reinterpret_cast<const float4v*>(cs + k + 4 * i);
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                sum += c[i >> 2][i & 3];
            }
        }
        if (q == 0) {
            lo_s = lo;
            lam_s = fmaxf(1e-4f, 0.25f * (sum / (float)K - lo));
        }
    }
    __syncthreads();
    const float lo = lo_s, lam = lam_s;
    for (int k = q; k < K; k += kUpdateThreads) {
        cs[k] = expf(-(cs[k] - lo) / lam);
    }
    __syncthreads();
    float wsum = 0.0f, acc = 0.0f;
    const float* mine = run + (q >> 1) * pitch + (q & 1);
    for (int k0 = 0; k0 < K; k0 += T) {
        if (q < 2 * H) {
            const int n = K - k0 < T ? K - k0 : T;
            for (int k = 0; k < n; k += 16) {
                float4v w[4];
                float v[16];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    w[i] = *reinterpret_cast<const float4v*>(cs + k0 + k + 4 * i);
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    v[i] = mine[2 * (k + i)];
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    wsum += w[i >> 2][i & 3];
                    acc += w[i >> 2][i & 3] * v[i];
                }
            }
        }
        if (k0 + T < K) {
            __syncthreads();
            put();
            __syncthreads();
            fetch(k0 + 2 * T);
        }
    }
    if (q < 2 * H) {
        mean[agent * 2 * H + q] = acc / wsum;
    }
}

void hcheck(hipError_t e, const char* what)
{
    if (e != hipSuccess) {
        throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
    }
}

template <typename T>
struct Dev {
    T* p = nullptr;
    std::size_t n = 0;
    Dev() = default;
    Dev(const Dev&) = delete;
    Dev& operator=(const Dev&) = delete;
    ~Dev()
    {
        if (p != nullptr) {
            (void)hipFree(p);
        }
    }
    void alloc(std::size_t count)
    {
        if (count <= n && p != nullptr) {
            return;
        }
        if (p != nullptr) {
            (void)hipFree(p);
            p = nullptr;
        }
        n = count;
        hcheck(hipMalloc(reinterpret_cast<void**>(&p), std::max<std::size_t>(1, count) * sizeof(T)), "hipMalloc");
    }
    void put(const T* host, std::size_t count)
    {
        alloc(count);
        hcheck(hipMemcpy(p, host, count * sizeof(T), hipMemcpyHostToDevice), "upload");
    }
};

} // namespace

using Rollout = void (*)(Desc, const float*, const float*, const unsigned*, float*, float*, u64, float, float, unsigned, unsigned);

namespace {

template <int NC, int Q>
Rollout rollout_of(int HB)
{
    static constexpr Rollout by_hidden[] = {k_mppi_rollout<1, NC, Q>, k_mppi_rollout<2, NC, Q>, k_mppi_rollout<3, NC, Q>,
        k_mppi_rollout<4, NC, Q>, k_mppi_rollout<5, NC, Q>, k_mppi_rollout<6, NC, Q>, k_mppi_rollout<7, NC, Q>, k_mppi_rollout<8, NC, Q>};
    static_assert(sizeof by_hidden / sizeof *by_hidden == kMaxWidth / 16, "every hidden width");
    return by_hidden[HB - 1];
}

} // namespace

struct fe_mppi {
    int F = 0, hid = 0, horizon = 0, samples = 0, HB = 0, NC = 0, fb = 0, lds = 0, cus = 1;
    Rollout rollout[2] = {};  // one, two tiles a wave
    int resident[2] = {1, 1}; // their waves the card holds at once
    bool dynamics = false, costed = false;
    Dev<half8> frags;
    Dev<float> tables;
    std::vector<float> host_tables;
    float action_weight = 0.0f;
    Dev<float> obs, mean, acts, cost;
    Dev<unsigned> ids;
    std::string error;
    // where the tables begin, in floats
    int b2() const { return hid; }
    int b3() const { return 2 * hid; }
    int shift() const { return b3() + 16 * fb; }
    int inscale() const { return shift() + 32 * NC; }
    int scale() const { return inscale() + 32 * NC; }
    int target() const { return scale() + 16 * fb; }
    int weight() const { return target() + 16 * fb; }
};

namespace {

int fail(fe_mppi* p, const std::string& what)
{
    if (p != nullptr) {
        p->error = what;
    }
    return -1;
}

// W[out][in] (row-major, fp32) as fragments: blocks of 16 outputs by 32 inputs, zero past both.
void pack(std::vector<_Float16>& to, const float* w, int out, int in, int blocks, int chunks)
{
    for (int ob = 0; ob < blocks; ++ob) {
        for (int c = 0; c < chunks; ++c) {
            for (int l = 0; l < 64; ++l) {
                for (int e = 0; e < 8; ++e) {
                    const int o = 16 * ob + l % 16, i = kfeat(c, l / 16, e);
                    to.push_back(static_cast<_Float16>(o < out && i < in ? w[static_cast<std::size_t>(o) * in + i] : 0.0f));
                }
            }
        }
    }
}

} // namespace

extern "C" {

fe_mppi* fe_mppi_create(int features, int hidden, int horizon, int samples, char* why, size_t why_bytes)
{
    auto say = [&](const std::string& s) {
        if (why != nullptr && why_bytes > 0) {
            std::snprintf(why, why_bytes, "%s", s.c_str());
        }
    };
    if (features < 1 || features + 2 > kMaxState || hidden < 16 || hidden > kMaxWidth || hidden % 16 != 0 || horizon < 1 || horizon > 64 ||
        samples < 16 || samples > 1024 || samples % 16 != 0) {
        say("features 1..62, hidden 16..128 (a multiple of 16), horizon 1..64, samples 16..1024 (a multiple of 16)");
        return nullptr;
    }
    fe_hip_device_info info{};
    if (fe_hip_device_open(&info) != 0) {
        say(std::string("no HIP device: ") + fe_hip_unavailable());
        return nullptr;
    }
    auto p = std::make_unique<fe_mppi>();
    p->cus = std::max(info.compute_units, 1);
    p->F = features;
    p->hid = hidden;
    p->horizon = horizon;
    p->samples = samples;
    p->HB = hidden / 16;
    p->NC = (features + 2 + 31) / 32;
    p->fb = (features + 15) / 16;
    p->lds = lds_bytes(p->HB, p->NC, p->fb);
    p->rollout[0] = p->NC == 1 ? rollout_of<1, 1>(p->HB) : rollout_of<2, 1>(p->HB);
    p->rollout[1] = p->NC == 1 ? rollout_of<1, 2>(p->HB) : rollout_of<2, 2>(p->HB);
    for (int q = 0; q < 2; ++q) {
        int blocks = 0;
        const void* k = reinterpret_cast<const void*>(p->rollout[q]);
        if ((p->lds > 64 * 1024 && hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, p->lds) != hipSuccess) ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, k, 256, static_cast<std::size_t>(p->lds)) != hipSuccess || blocks < 1) {
            say("the rollout does not fit the card");
            return nullptr;
        }
        p->resident[q] = 4 * blocks * p->cus;
    }
    p->host_tables.assign(static_cast<std::size_t>(4 * table_count(p->HB, p->NC, p->fb)), 0.0f);
    return p.release();
}

void fe_mppi_free(fe_mppi* p) { delete p; }
const char* fe_mppi_error(fe_mppi* p) { return p != nullptr ? p->error.c_str() : "no planner"; }

int fe_mppi_set_dynamics(fe_mppi* p, const float* weights, const float* in_shift, const float* in_scale, const float* scale)
{
    if (p == nullptr || weights == nullptr || in_shift == nullptr || in_scale == nullptr || scale == nullptr) {
        return fail(p, "invalid arguments");
    }
    try {
        const int F = p->F, I = F + 2, Hd = p->hid;
        const float* w1 = weights;
        const float* b1 = w1 + static_cast<std::size_t>(I) * Hd;
        const float* w2 = b1 + Hd;
        const float* b2 = w2 + static_cast<std::size_t>(Hd) * Hd;
        const float* w3 = b2 + Hd;
        const float* b3 = w3 + static_cast<std::size_t>(Hd) * F;
        std::vector<_Float16> packed;
        packed.reserve(static_cast<std::size_t>(frag_count(p->HB, p->NC, p->fb)) * 512);
        const int HC = (p->HB + 1) / 2;
        pack(packed, w1, Hd, I, p->HB, p->NC);
        pack(packed, w2, Hd, Hd, p->HB, HC);
        pack(packed, w3, F, Hd, p->fb, HC);
        p->frags.put(reinterpret_cast<const half8*>(packed.data()), packed.size() / 8);
        float* to = p->host_tables.data();
        std::copy(b1, b1 + Hd, to);
        std::copy(b2, b2 + Hd, to + p->b2());
        std::copy(b3, b3 + F, to + p->b3());
        std::copy(in_shift, in_shift + I, to + p->shift());
        std::copy(in_scale, in_scale + I, to + p->inscale());
        std::copy(scale, scale + F, to + p->scale());
        p->tables.put(to, p->host_tables.size());
        p->dynamics = true;
        return 0;
    } catch (const std::exception& e) {
        return fail(p, e.what());
    }
}

int fe_mppi_set_cost(fe_mppi* p, const float* target, const float* weight, float action_weight)
{
    if (p == nullptr || target == nullptr || weight == nullptr) {
        return fail(p, "invalid arguments");
    }
    try {
        std::copy(target, target + p->F, p->host_tables.data() + p->target());
        std::copy(weight, weight + p->F, p->host_tables.data() + p->weight());
        p->tables.put(p->host_tables.data(), p->host_tables.size());
        p->action_weight = action_weight;
        p->costed = true;
        return 0;
    } catch (const std::exception& e) {
        return fail(p, e.what());
    }
}

int fe_mppi_plan(fe_mppi* p, int agents, const float* obs, const uint32_t* ids, uint64_t tick, float sigma, float dt, float* mean,
    float* cost_out)
{
    if (p == nullptr || agents < 1 || obs == nullptr || ids == nullptr || mean == nullptr) {
        return fail(p, "invalid arguments");
    }
    if (!p->dynamics || !p->costed) {
        return fail(p, "set the dynamics and the cost first");
    }
    try {
        const int F = p->F, H = p->horizon, K = p->samples;
        const long long tiles = static_cast<long long>(agents) * (K / 16);
        // Two tiles a wave share the weights' reads and hide each other's latency, once there are four a SIMD: hidden 64,
        // 128 and 16 take 205, 315, 137 us a plan against one tile's 200, 328, 136 at four a SIMD, 307, 546, 181 against 316,
        // 588, 187 at eight; at three one tile is the faster (174, 258, 123 against 203, 310, 135), and for a lone agent (121
        // against 146).
        const int two = tiles >= 16LL * p->cus && K > 16 ? 1 : 0;
        const unsigned per_agent = static_cast<unsigned>((K / 16 + two) / (1 + two));
        const long long items = static_cast<long long>(agents) * per_agent;
        if (items >= 4294967296LL - 2097152) { // the kernel's index, and its stride past the end; their actions would be 550 GB
            return fail(p, "too many agents for one plan");
        }
        // one round of blocks, each wave as many items as any other, where more of them would start a second round
        const long long rounds = (items + p->resident[two] - 1) / p->resident[two];
        const long long waves = (items + rounds - 1) / rounds;
        const hipStream_t s = static_cast<hipStream_t>(fe_hip_stream());
        p->obs.put(obs, static_cast<std::size_t>(agents) * F);
        p->ids.put(ids, static_cast<std::size_t>(agents));
        p->mean.put(mean, static_cast<std::size_t>(agents) * H * 2);
        p->acts.alloc(static_cast<std::size_t>(agents) * K * H * 2);
        p->cost.alloc(static_cast<std::size_t>(agents) * K);
        const Desc d{F, p->fb, H, K, p->frags.p, reinterpret_cast<const float4v*>(p->tables.p), p->action_weight};
        hipLaunchKernelGGL(p->rollout[two], dim3(static_cast<unsigned>((waves + 3) / 4)), dim3(256), static_cast<unsigned>(p->lds), s, d, p->obs.p,
            p->mean.p, p->ids.p, p->acts.p, p->cost.p, static_cast<unsigned long long>(tick), sigma, dt, static_cast<unsigned>(items), per_agent);
        hipLaunchKernelGGL(k_mppi_update, dim3(static_cast<unsigned>(agents)), dim3(kUpdateThreads), 0, s, p->cost.p, p->acts.p, p->mean.p, K, H);
        hcheck(hipGetLastError(), "mppi launch");
        hcheck(hipMemcpyAsync(mean, p->mean.p, sizeof(float) * static_cast<std::size_t>(agents) * H * 2, hipMemcpyDeviceToHost, s), "download");
        if (cost_out != nullptr) {
            hcheck(hipMemcpyAsync(cost_out, p->cost.p, sizeof(float) * static_cast<std::size_t>(agents) * K, hipMemcpyDeviceToHost, s), "download");
        }
        hcheck(hipStreamSynchronize(s), "sync");
        return 0;
    } catch (const std::exception& e) {
        return fail(p, e.what());
    }
}

} // extern "C"
