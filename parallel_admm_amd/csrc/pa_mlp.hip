// MLP forward, backward and Adam on MFMA (gfx950, v_mfma_f32_16x16x32_bf16).
//
// A pass is one launch (inference) or three (a training step): k_mlp takes 32
// rows per workgroup through the whole network and back, k_weight_grads forms
// every weight gradient, k_reduce sums its splits and takes the Adam step.
// Every product is an "NT" one, C[M][N] = sum_k A[m][k] Bt[n][k], with both
// operands BF16 and K contiguous, FP32 accumulation and 16x16 output tiles:
//   forward hidden  a = C + b, H = SiLU(a) (H^T and SiLU'(a) when training)
//   forward output  y = C + b, dY = (y - t) / n, loss partials
//   backward        dA = C * SiLU'(a)  (and dA^T)
//   weight grads    split-K partials of dA^T H (bias gradient via a ones row)
// Partial weight gradients are summed in a fixed order, so a training run is
// bit-reproducible.
#include "pa_mlp.hpp"

#include <algorithm>
#include <cmath>
#include <numeric>
#include <mutex>
#include <random>
#include <string>

namespace pa {
namespace {

using namespace mlp;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline uint16_t to_bf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

__device__ inline bf16x8 frag(const uint16_t* p) { return *reinterpret_cast<const bf16x8*>(p); }
// Four BF16 values of consecutive rows of one column into a transposed array.
__device__ inline void put4(uint16_t* p, const uint16_t (&v)[4]) {
    *reinterpret_cast<uint2*>(p) = make_uint2((uint32_t)v[0] | (uint32_t)v[1] << 16, (uint32_t)v[2] | (uint32_t)v[3] << 16);
}

struct MlpArgs {
    const float* src; // rows of `stride` floats: features, then 2 targets when training; via idx when given
    int stride;
    const int32_t* idx;
    int n, cap; // real rows; leading dimension of the transposed arrays
    const uint16_t *W1p, *W2, *W3, *W4p, *W2T, *W3T, *W4T;
    const float* w; // FP32 parameters (biases)
    float* Y;       // [rows][2]
    // training only
    uint16_t *XT, *H1T, *H2T, *H3T, *dYT, *dA1T, *dA2T, *dA3T;
    double* loss_part;
    float inv_n;
};

// 32 rows through the network, and with TRAIN back.  A layer over 8192 rows is
// 0.27 GFLOP, under a microsecond of MFMA, so as launches of their own (12 of
// 5-9 us in a training step) the layers cost only their latency; here
// activations pass from layer to layer through LDS and SiLU' stays in
// registers.  Wave w owns columns 32 w .. 32 w + 31 of every hidden layer in
// both directions (2 x 2 tiles), so the SiLU' of its forward tiles is where its
// backward tiles need it.  A layer's weight fragments come straight from L2,
// one layer ahead of their use.
// Fragment layout of the 16x16x32 product: lane l holds row (l % 16) of A and
// column (l % 16) of B at k = 8 (l / 16) .. +7; the accumulator of lane l
// holds column l % 16, rows 4 (l / 16) .. +3.
// Training step of 8192 rows: 15.4 us for this and 14.2 us for the weight
// gradients, against 64 and 33 us as one launch per product.
constexpr int FR = 32;         // rows per workgroup
constexpr int AST = H + 8;     // LDS row strides (BF16): 16-byte aligned rows on rotating banks
constexpr int XST = INP + 8;
template <bool TRAIN> __global__ void __launch_bounds__(256) k_mlp(MlpArgs g) {
    __shared__ __align__(16) uint16_t act[2][FR * AST];
    __shared__ __align__(16) uint16_t xin[FR * XST]; // the input, then dY
    __shared__ float tgt[FR][OUT];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, r16 = lane & 15, kq = (lane >> 4) * 8, rq = (lane >> 4) * 4;
    const int tiles = gridDim.x, tile = tiles % 8 ? blockIdx.x : (blockIdx.x % 8) * (tiles / 8) + blockIdx.x / 8; // an XCD's tiles adjoin
    const int row0 = tile * FR;
    const int col[2] = {32 * wave + r16, 32 * wave + 16 + r16};
    // the input rows (BF16, zero padded) and the targets
    for (int e = t; e < FR * INP; e += 256) {
        const int s = e / INP, k = e % INP, r = row0 + s;
        float v = 0.f;
        if (r < g.n && k < IN) v = g.src[(size_t)(g.idx ? g.idx[r] : r) * g.stride + k];
        xin[s * XST + k] = to_bf16(v);
    }
    if (TRAIN && t < FR * OUT) {
        const int s = t / OUT, r = row0 + s;
        tgt[s][t % OUT] = r < g.n ? g.src[(size_t)(g.idx ? g.idx[r] : r) * g.stride + IN + t % OUT] : 0.f;
    }
    bf16x8 w[2][4], wn[2][4];
    auto load = [&](bf16x8(&o)[2][4], const uint16_t* W, int ld, int steps) {
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (k < steps) o[c][k] = frag(W + (size_t)col[c] * ld + 32 * k + kq);
    };
    f32x4 acc[2][2]; // [row tile][column tile]
    auto product = [&](const bf16x8(&b)[2][4], const uint16_t* A, int st, int steps) {
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int c = 0; c < 2; c++) acc[m][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (k < steps)
#pragma unroll
                for (int m = 0; m < 2; m++) {
                    const bf16x8 a = frag(A + (16 * m + r16) * st + 32 * k + kq);
#pragma unroll
                    for (int c = 0; c < 2; c++) acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[c][k], acc[m][c], 0, 0, 0);
                }
    };
    float S[3][2][2][4]; // SiLU' of the wave's tiles
    auto silu = [&](int l, const float* bias, uint16_t* out, uint16_t* outT) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const float bc = bias[col[c]];
#pragma unroll
            for (int m = 0; m < 2; m++) {
                uint16_t hb[4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float a = acc[m][c][r] + bc;
                    const float sg = 1.f / (1.f + __expf(-a));
                    hb[r] = to_bf16(a * sg);
                    out[(16 * m + rq + r) * AST + col[c]] = hb[r];
                    if (TRAIN) S[l][m][c][r] = sg * (1.f + a * (1.f - sg));
                }
                if (TRAIN) put4(outT + (size_t)col[c] * g.cap + row0 + 16 * m + rq, hb);
            }
        }
    };
    load(w, g.W1p, INP, 1);
    load(wn, g.W2, H, 4);
    __syncthreads();
    if (TRAIN)
        for (int e = t; e < INA * FR; e += 256) { // X^T, row 10 = 1 on real rows
            const int k = e / FR, s = e % FR;
            g.XT[(size_t)k * g.cap + row0 + s] = k < IN ? xin[s * XST + k] : to_bf16(k == IN && row0 + s < g.n ? 1.f : 0.f);
        }
    product(w, xin, XST, 1);
    silu(0, g.w + OB1, act[0], g.H1T);
    load(w, g.W3, H, 4);
    __syncthreads();
    product(wn, act[0], AST, 4);
    silu(1, g.w + OB2, act[1], g.H2T);
    if (TRAIN) load(wn, g.W4T, OUTK, 1);
    bf16x8 w4[4]; // output layer: wave m < 2 takes row tile m
#pragma unroll
    for (int k = 0; k < 4; k++) w4[k] = frag(g.W4p + (size_t)r16 * H + 32 * k + kq);
    __syncthreads();
    product(w, act[1], AST, 4);
    silu(2, g.w + OB3, act[0], g.H3T);
    if (TRAIN) {
        load(w, g.W3T, H, 4);
        for (int e = t; e < FR * XST; e += 256) xin[e] = 0; // becomes dY: its last reader passed two barriers ago
    }
    __syncthreads();
    if (wave < 2) {
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 4; k++) o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(act[0] + (16 * wave + r16) * AST + 32 * k + kq), w4[k], o, 0, 0, 0);
        double l = 0.0;
        if (r16 < OUT) {
            const float bc = g.w[OB4 + r16];
            uint16_t eb[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int s = 16 * wave + rq + r, row = row0 + s;
                const float y = o[r] + bc;
                g.Y[(size_t)row * OUT + r16] = y;
                if (TRAIN) {
                    const float e = row < g.n ? y - tgt[s][r16] : 0.f;
                    l += (double)e * (double)e;
                    eb[r] = to_bf16(e * g.inv_n);
                    xin[s * XST + r16] = eb[r];
                }
            }
            if (TRAIN) put4(g.dYT + (size_t)r16 * g.cap + row0 + 16 * wave + rq, eb);
        }
        if (TRAIN) {
            for (int q = 32; q > 0; q >>= 1) l += __shfl_xor(l, q);
            if (lane == 0) g.loss_part[2 * tile + wave] = l;
        }
    }
    if constexpr (TRAIN) {
        auto back = [&](int l, uint16_t* out, uint16_t* outT) {
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int m = 0; m < 2; m++) {
                    uint16_t vb[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        vb[r] = to_bf16(acc[m][c][r] * S[l][m][c][r]);
                        if (out) out[(16 * m + rq + r) * AST + col[c]] = vb[r];
                    }
                    put4(outT + (size_t)col[c] * g.cap + row0 + 16 * m + rq, vb);
                }
        };
        __syncthreads();
        product(wn, xin, XST, 1);
        back(2, act[1], g.dA3T);
        load(wn, g.W2T, H, 4);
        __syncthreads();
        product(w, act[1], AST, 4);
        back(1, act[0], g.dA2T);
        __syncthreads();
        product(wn, act[0], AST, 4);
        back(0, nullptr, g.dA1T);
    }
}

// Every weight gradient in one launch: split-K partials of dA^T H, one 16x16
// tile and split per wave.  A layer's tiles start at first[l]; a wave's
// fragments of eight K steps are in flight at once (14.2 us at 8192 rows; four
// launches with one step at a time 33).  Workgroups of a split share an XCD, so an
// L2 reads one eighth of the 7 MB that k_mlp left, mostly rows written there.
struct GradArgs {
    const uint16_t* A[4];
    const uint16_t* Bt[4];
    float* out[4];
    int M[4], N[4], first[5];
    int splits, per, cap; // K steps (32 rows) per split
};
__global__ void __launch_bounds__(256) k_weight_grads(GradArgs g) {
    const int lane = threadIdx.x & 63;
    const int s8 = min(g.splits, 8), ns = g.splits / s8; // splits are powers of two up to 16
    const int split = (blockIdx.x % s8) * ns + (blockIdx.x / s8) % ns, t = (blockIdx.x / g.splits) * 4 + (threadIdx.x >> 6);
    if (t >= g.first[4]) return;
    int l = 0;
    while (t >= g.first[l + 1]) l++;
    const int tn_count = g.N[l] >> 4, q = t - g.first[l], tm = q / tn_count, tn = q - tm * tn_count;
    const int r16 = lane & 15, kq = (lane >> 4) * 8;
    const size_t k0 = (size_t)split * g.per * 32 + kq;
    const uint16_t* pa = g.A[l] + (size_t)(tm * 16 + r16) * g.cap + k0;
    const uint16_t* pb = g.Bt[l] + (size_t)(tn * 16 + r16) * g.cap + k0;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < g.per; s += 8) {
        bf16x8 a[8], b[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const size_t k = 32 * (size_t)min(s + u, g.per - 1);
            a[u] = frag(pa + k);
            b[u] = frag(pb + k);
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (s + u < g.per) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u], b[u], acc, 0, 0, 0);
    }
    float* o = g.out[l] + ((size_t)split * g.M[l] + tm * 16 + (lane >> 4) * 4) * g.N[l] + tn * 16 + r16;
#pragma unroll
    for (int r = 0; r < 4; r++) o[(size_t)r * g.N[l]] = acc[r];
}

struct Copies {
    uint16_t *W1p, *W2, *W2T, *W3, *W3T, *W4p, *W4T;
};

__device__ inline void write_copies(const Copies& c, int p, float val) {
    const uint16_t b = to_bf16(val);
    if (p < OB1) {
        c.W1p[(p / IN) * INP + p % IN] = b;
    } else if (p >= OW2 && p < OB2) {
        const int q = p - OW2, r = q / H, k = q % H;
        c.W2[r * H + k] = b;
        c.W2T[k * H + r] = b;
    } else if (p >= OW3 && p < OB3) {
        const int q = p - OW3, r = q / H, k = q % H;
        c.W3[r * H + k] = b;
        c.W3T[k * H + r] = b;
    } else if (p >= OW4 && p < OB4) {
        const int q = p - OW4, r = q / H, k = q % H;
        c.W4p[r * H + k] = b;
        c.W4T[k * OUTK + r] = b;
    }
}

__global__ void k_refresh(const float* __restrict__ w, Copies c) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < NPARAM) write_copies(c, p, w[p]);
}

// Gradient of parameter p = sum over splits of its partial (fixed order);
// mode 0 stores it, mode 1 applies Adam (Kingma and Ba, ICLR 2015) with bias
// corrections bc1 = 1 - beta1^t, bc2 = 1 - beta2^t and refreshes the BF16 copies.
__global__ void k_reduce(int mode, int splits, const float* __restrict__ part, int64_t off2, int64_t off3, int64_t off4, float lr,
                         float bc1, float bc2, float* __restrict__ w, float* __restrict__ m, float* __restrict__ v,
                         float* __restrict__ grad, Copies c) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= NPARAM) return;
    const float* base;
    int rows, cols, r, k;
    if (p < OW2) {
        base = part;
        rows = H;
        cols = INA;
        if (p < OB1) r = p / IN, k = p % IN;
        else r = p - OB1, k = IN;
    } else if (p < OW3) {
        base = part + off2;
        rows = H;
        cols = HA;
        if (p < OB2) r = (p - OW2) / H, k = (p - OW2) % H;
        else r = p - OB2, k = H;
    } else if (p < OW4) {
        base = part + off3;
        rows = H;
        cols = HA;
        if (p < OB3) r = (p - OW3) / H, k = (p - OW3) % H;
        else r = p - OB3, k = H;
    } else {
        base = part + off4;
        rows = OUTP;
        cols = HA;
        if (p < OB4) r = (p - OW4) / H, k = (p - OW4) % H;
        else r = p - OB4, k = H;
    }
    float gsum = 0.f;
    for (int s = 0; s < splits; s += 8) { // at most 16 splits, eight loads in flight
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = base[((size_t)min(s + u, splits - 1) * rows + r) * cols + k];
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (s + u < splits) gsum += v[u];
    }
    if (mode == 0) {
        grad[p] = gsum;
        return;
    }
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float mm = b1 * m[p] + (1.f - b1) * gsum;
    const float vv = b2 * v[p] + (1.f - b2) * gsum * gsum;
    m[p] = mm;
    v[p] = vv;
    const float wn = w[p] - lr * (mm / bc1) / (sqrtf(vv / bc2) + eps);
    w[p] = wn;
    write_copies(c, p, wn);
}

// Row 128 of every transposed hidden buffer is 1 (bias gradient), rows above are 0.
__global__ void k_ones_rows(int cap, uint16_t* __restrict__ a, uint16_t* __restrict__ b, uint16_t* __restrict__ c) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= cap) return;
    const uint16_t one = to_bf16(1.f);
    a[(size_t)H * cap + s] = one;
    b[(size_t)H * cap + s] = one;
    c[(size_t)H * cap + s] = one;
}

// ---------------------------------------------------------------------------
// Scratch of the forward pass that allocates nothing (pa_mlp_forward_noalloc):
// one file-scope device array per GPU of the size that the C ABI states, holding
// the staged input (float [rows][10]) and the output (float [rows][2]) of up to
// kNoAllocRows padded rows; activations stay on chip.  Every byte a call reads
// is written earlier in the same call, so nothing is cleared between calls.
// Calls that overlap on one GPU share the array and race; calls on different
// GPUs use each GPU's own copy.
// ---------------------------------------------------------------------------
constexpr size_t kSy = (size_t)kNoAllocRows * IN * sizeof(float);
static_assert(kSy % 256 == 0 && kSy + (size_t)kNoAllocRows * OUT * sizeof(float) == kNoAllocScratchBytes, "scratch layout and size differ");

__device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

// Device address of `scratch` on each device, resolved once per device with
// that device current (the array's name in host code is only a stand-in).
std::mutex g_scratch_mu;
void* g_scratch_ptr[64] = {};

void* scratch_address() {
    int dev = 0;
    PA_HIP(hipGetDevice(&dev));
    PA_CHECK(dev >= 0 && dev < 64, PA_ERR_INVALID, "mlp: device ordinal beyond the scratch table");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        PA_CHECK(e == hipSuccess && ptr, PA_ERR_HIP,
                 std::string("mlp: hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
        g_scratch_ptr[dev] = ptr;
    }
    return g_scratch_ptr[dev];
}

} // namespace

Mlp::Mlp(hipStream_t s) : Mlp(Empty{}) {
    if (s) {
        stream = s;
    } else {
        PA_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
        own_stream = true;
    }
    (void)scratch_address(); // set-up of the allocation-free forward on this device
    w.alloc(NPARAM);
    adam_m.alloc(NPARAM);
    adam_v.alloc(NPARAM);
    grad.alloc(NPARAM);
    W1p.alloc(H * INP);
    W2.alloc(H * H);
    W2T.alloc(H * H);
    W3.alloc(H * H);
    W3T.alloc(H * H);
    W4p.alloc(OUTP * H);
    W4T.alloc(H * OUTK);
    for (DBuf<uint16_t>* b : {&W1p, &W4p, &W4T}) b->zero(stream);
    adam_m.zero(stream);
    adam_v.zero(stream);
    PA_HIP(hipStreamSynchronize(stream));
}

Mlp::~Mlp() {
    if (stream) (void)hipStreamSynchronize(stream);
    if (own_stream && stream) (void)hipStreamDestroy(stream);
}

void Mlp::init_params(uint64_t seed) {
    std::mt19937_64 rng(seed);
    std::vector<float> h(NPARAM);
    auto fill = [&](int off, int count, int fan_in) {
        const double a = 1.0 / std::sqrt((double)fan_in);
        std::uniform_real_distribution<double> u(-a, a);
        for (int i = 0; i < count; i++) h[off + i] = (float)u(rng);
    };
    fill(OW1, H * IN, IN);
    fill(OB1, H, IN);
    fill(OW2, H * H, H);
    fill(OB2, H, H);
    fill(OW3, H * H, H);
    fill(OB3, H, H);
    fill(OW4, OUT * H, H);
    fill(OB4, OUT, H);
    set_params(h.data());
}

void Mlp::set_params(const float* host) {
    w.upload(host, NPARAM, stream);
    adam_m.zero(stream);
    adam_v.zero(stream);
    adam_t = 0;
    Copies c{W1p.p, W2.p, W2T.p, W3.p, W3T.p, W4p.p, W4T.p};
    hipLaunchKernelGGL(k_refresh, dim3(grid_for(NPARAM, 256)), dim3(256), 0, stream, (const float*)w.p, c);
    PA_LAUNCH_CHECK();
    PA_HIP(hipStreamSynchronize(stream));
}

void Mlp::get_params(float* host) {
    w.download(host, NPARAM, stream);
    PA_HIP(hipStreamSynchronize(stream));
}

float* Mlp::outputs(int rows) {
    PA_CHECK(rows > 0 && rows % 32 == 0, PA_ERR_INVALID, "mlp: rows must be a positive multiple of 32");
    if ((size_t)rows * OUT > Y.n) Y.alloc(std::max((size_t)rows * OUT, Y.n + Y.n / 2));
    return Y.p;
}

void Mlp::ensure(int rows) {
    outputs(rows);
    if (rows <= cap) return;
    cap = 0; // until everything below is in place
    const size_t c = (size_t)rows;
    XT.alloc(c * INA);
    for (DBuf<uint16_t>* b : {&H1T, &H2T, &H3T}) b->alloc(c * HA);
    for (DBuf<uint16_t>* b : {&dA1T, &dA2T, &dA3T}) b->alloc(c * H);
    dYT.alloc(c * OUTP);
    part.alloc((size_t)16 * (2 * H * HA + H * INA + OUTP * HA)); // up to 16 splits
    for (DBuf<uint16_t>* b : {&H1T, &H2T, &H3T, &dYT}) b->zero(stream);
    hipLaunchKernelGGL(k_ones_rows, dim3(grid_for(rows, 256)), dim3(256), 0, stream, rows, H1T.p, H2T.p, H3T.p);
    PA_LAUNCH_CHECK();
    PA_HIP(hipStreamSynchronize(stream));
    cap = rows;
}

static MlpArgs mlp_args(const Mlp& m, const float* src, int stride, const int32_t* idx, int n, float* y) {
    MlpArgs g{};
    g.src = src;
    g.stride = stride;
    g.idx = idx;
    g.n = n;
    g.W1p = m.W1p.p;
    g.W2 = m.W2.p;
    g.W3 = m.W3.p;
    g.W4p = m.W4p.p;
    g.w = m.w.p;
    g.Y = y;
    return g;
}

void Mlp::infer(const float* src, int stride, int n, int rows, float* y) {
    PA_CHECK(rows > 0 && rows % FR == 0 && n >= 0 && n <= rows, PA_ERR_INVALID, "mlp: bad forward shape");
    hipLaunchKernelGGL(k_mlp<false>, dim3(rows / FR), dim3(256), 0, stream, mlp_args(*this, src, stride, nullptr, n, y));
    PA_LAUNCH_CHECK();
}

void Mlp::train_pass(const float* src, int stride, const int32_t* idx, int n, int rows, double* loss_out) {
    PA_CHECK(rows > 0 && rows <= cap && rows % FR == 0 && n >= 0 && n <= rows, PA_ERR_INVALID, "mlp: bad training shape");
    MlpArgs a = mlp_args(*this, src, stride, idx, n, Y.p);
    a.cap = cap;
    a.W2T = W2T.p;
    a.W3T = W3T.p;
    a.W4T = W4T.p;
    a.XT = XT.p;
    a.H1T = H1T.p;
    a.H2T = H2T.p;
    a.H3T = H3T.p;
    a.dYT = dYT.p;
    a.dA1T = dA1T.p;
    a.dA2T = dA2T.p;
    a.dA3T = dA3T.p;
    a.loss_part = loss_out;
    a.inv_n = n > 0 ? 1.f / (float)n : 0.f;
    hipLaunchKernelGGL(k_mlp<true>, dim3(rows / FR), dim3(256), 0, stream, a);
    PA_LAUNCH_CHECK();
    const int slabs = rows / 32;
    splits = 16;
    while (slabs % splits) splits /= 2;
    const int64_t off2 = (int64_t)splits * H * INA, off3 = off2 + (int64_t)splits * H * HA, off4 = off3 + (int64_t)splits * H * HA;
    // layers 4 to 1: dW4 = dY^T H3, dW3 = dA3^T H2, dW2 = dA2^T H1, dW1 = dA1^T X
    GradArgs g{{dYT.p, dA3T.p, dA2T.p, dA1T.p}, {H3T.p, H2T.p, H1T.p, XT.p}, {part.p + off4, part.p + off3, part.p + off2, part.p},
               {OUTP, H, H, H}, {HA, HA, HA, INA}, {0, 0, 0, 0, 0}, splits, slabs / splits, cap};
    for (int l = 0; l < 4; l++) g.first[l + 1] = g.first[l] + (g.M[l] / 16) * (g.N[l] / 16);
    hipLaunchKernelGGL(k_weight_grads, dim3((g.first[4] + 3) / 4 * splits), dim3(256), 0, stream, g);
    PA_LAUNCH_CHECK();
}

void Mlp::reduce(int mode, float lr) {
    const int64_t off2 = (int64_t)splits * H * INA, off3 = off2 + (int64_t)splits * H * HA, off4 = off3 + (int64_t)splits * H * HA;
    float bc1 = 1.f, bc2 = 1.f;
    if (mode == 1) {
        adam_t++;
        bc1 = (float)(1.0 - std::pow(0.9, adam_t));
        bc2 = (float)(1.0 - std::pow(0.999, adam_t));
    }
    Copies c{W1p.p, W2.p, W2T.p, W3.p, W3T.p, W4p.p, W4T.p};
    hipLaunchKernelGGL(k_reduce, dim3(grid_for(NPARAM, 256)), dim3(256), 0, stream, mode, splits, (const float*)part.p, off2, off3, off4, lr,
                       bc1, bc2, w.p, adam_m.p, adam_v.p, grad.p, c);
    PA_LAUNCH_CHECK();
}

// Sum of the loss partials of `rows` rows, in row order.
double Mlp::loss(int rows) {
    std::vector<double> h(rows / 16);
    loss_part.download(h.data(), h.size(), stream);
    PA_HIP(hipStreamSynchronize(stream));
    double s = 0;
    for (double v : h) s += v;
    return s;
}

void Mlp::forward_host(const float* x, int n, float* y) {
    PA_CHECK(n > 0, PA_ERR_INVALID, "mlp: no rows");
    const int rows = pad_rows(n);
    samples.reserve((size_t)n * IN);
    samples.upload(x, (size_t)n * IN, stream);
    infer(samples.p, IN, n, rows, outputs(rows));
    Y.download(y, (size_t)n * OUT, stream);
    PA_HIP(hipStreamSynchronize(stream));
}

// The same forward as forward_host with input and output in the file-scope
// scratch array: no device memory is allocated or freed.
void Mlp::forward_noalloc(const float* x, int n, float* y) {
    PA_CHECK(n > 0, PA_ERR_INVALID, "mlp: no rows");
    PA_CHECK(n <= kNoAllocRows, PA_ERR_INVALID,
             "mlp: the allocation-free forward takes at most " + std::to_string(kNoAllocRows) + " rows per call");
    const int rows = pad_rows(n);
    unsigned char* base = static_cast<unsigned char*>(scratch_address());
    float* xin = reinterpret_cast<float*>(base);
    float* yo = reinterpret_cast<float*>(base + kSy);
    PA_HIP(hipMemcpyAsync(xin, x, sizeof(float) * (size_t)n * IN, hipMemcpyHostToDevice, stream));
    infer(xin, IN, n, rows, yo);
    PA_HIP(hipMemcpyAsync(y, yo, sizeof(float) * (size_t)n * OUT, hipMemcpyDeviceToHost, stream));
    PA_HIP(hipStreamSynchronize(stream));
}

static void stage_xt(DBuf<float>& buf, const float* x, const float* t, int n, hipStream_t s) {
    std::vector<float> h((size_t)n * (IN + OUT));
    for (int i = 0; i < n; i++) {
        std::copy(x + (size_t)i * IN, x + (size_t)(i + 1) * IN, h.begin() + (size_t)i * (IN + OUT));
        h[(size_t)i * (IN + OUT) + IN] = t[2 * (size_t)i];
        h[(size_t)i * (IN + OUT) + IN + 1] = t[2 * (size_t)i + 1];
    }
    buf.reserve(h.size());
    buf.upload(h.data(), h.size(), s);
}

double Mlp::gradients_host(const float* x, const float* t, int n, float* g) {
    PA_CHECK(n > 0, PA_ERR_INVALID, "mlp: no rows");
    const int rows = pad_rows(n);
    ensure(rows);
    stage_xt(samples, x, t, n, stream);
    loss_part.reserve(rows / 16);
    train_pass(samples.p, IN + OUT, nullptr, n, rows, loss_part.p);
    reduce(0, 0.f);
    grad.download(g, NPARAM, stream);
    return loss(rows) / (2.0 * n);
}

double Mlp::adam_host(const float* x, const float* t, int n, float lr) {
    PA_CHECK(n > 0, PA_ERR_INVALID, "mlp: no rows");
    const int rows = pad_rows(n);
    ensure(rows);
    stage_xt(samples, x, t, n, stream);
    loss_part.reserve(rows / 16);
    train_pass(samples.p, IN + OUT, nullptr, n, rows, loss_part.p);
    const double l = loss(rows) / (2.0 * n);
    reduce(1, lr);
    PA_HIP(hipStreamSynchronize(stream));
    return l;
}

void Mlp::train_host(const float* samples_h, int64_t n, int epochs, int batch, float lr, uint64_t seed, double* epoch_loss) {
    PA_CHECK(n > 0 && n <= (int64_t)1 << 30 && epochs >= 1 && batch >= 32 && batch % 32 == 0, PA_ERR_INVALID,
             "mlp: bad training arguments");
    samples.reserve((size_t)n * (IN + OUT));
    samples.upload(samples_h, (size_t)n * (IN + OUT), stream);
    perm.reserve((size_t)n);
    ensure(batch);
    std::vector<int32_t> order((size_t)n);
    std::iota(order.begin(), order.end(), 0);
    std::mt19937_64 rng(seed);
    std::shuffle(order.begin(), order.end(), rng);
    // an epoch's loss partials stay on the device until its end: no wait per batch
    const size_t per_batch = (size_t)batch / 16;
    std::vector<double> h(((size_t)n + batch - 1) / batch * per_batch);
    loss_part.reserve(h.size());
    for (int e = 0; e < epochs; e++) {
        perm.upload(order.data(), order.size(), stream);
        size_t k = 0;
        for (int64_t b0 = 0; b0 < n; b0 += batch, k++) {
            const int nb = (int)std::min<int64_t>(batch, n - b0);
            train_pass(samples.p, IN + OUT, perm.p + b0, nb, pad_rows(nb), loss_part.p + k * per_batch);
            reduce(1, lr);
        }
        if (e + 1 < epochs) std::shuffle(order.begin(), order.end(), rng); // the next epoch's order, beside this one's kernels
        loss_part.download(h.data(), k * per_batch, stream);
        PA_HIP(hipStreamSynchronize(stream));
        double lsum = 0;
        k = 0;
        for (int64_t b0 = 0; b0 < n; b0 += batch, k++) {
            const int parts = pad_rows((int)std::min<int64_t>(batch, n - b0)) / 16;
            double l = 0;
            for (int q = 0; q < parts; q++) l += h[k * per_batch + q];
            lsum += l / 2.0;
        }
        if (epoch_loss) epoch_loss[e] = lsum / (double)n;
    }
}

double Mlp::time_ms(int which, int rows, int reps) {
    PA_CHECK(reps > 0 && reps <= 100000 && (which == 0 || which == 1), PA_ERR_INVALID, "mlp: bad timing request");
    rows = pad_rows(rows);
    if (which == 0) outputs(rows);
    else ensure(rows);
    // a fixed synthetic batch: zero features and targets (timing only)
    samples.reserve((size_t)rows * (IN + OUT));
    PA_HIP(hipMemsetAsync(samples.p, 0, sizeof(float) * (size_t)rows * (IN + OUT), stream));
    loss_part.reserve(rows / 16);
    std::vector<float> keep(NPARAM);
    get_params(keep.data());
    hipEvent_t e0, e1;
    PA_HIP(hipEventCreate(&e0));
    PA_HIP(hipEventCreate(&e1));
    auto one = [&]() {
        if (which == 0) {
            infer(samples.p, IN + OUT, rows, rows, Y.p);
        } else {
            train_pass(samples.p, IN + OUT, nullptr, rows, rows, loss_part.p);
            reduce(1, 0.f);
        }
    };
    one();
    PA_HIP(hipEventRecord(e0, stream));
    for (int r = 0; r < reps; r++) one();
    PA_HIP(hipEventRecord(e1, stream));
    PA_HIP(hipEventSynchronize(e1));
    float ms = 0;
    PA_HIP(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    set_params(keep.data()); // the weights as before; the Adam state starts over
    return ms / reps;
}

} // namespace pa
