// Kernels of the warm-start network (layout and parameter vector in mlp.h).
//
// One wavefront evaluates 16 samples at a time on the matrix cores. Lane
// l = 16*g + c (g = l / 16, c = l % 16). With the 16x16x16 BF16 instruction:
//   A operand (weights, 16 rows x 16 k): row c, k = 4g..4g+3
//   B operand (activations, 16 k x 16 samples): k = 4g..4g+3, sample c
//   accumulator: rows 4g..4g+3, sample c
// so a layer's accumulator, after the activation and conversion to BF16, is
// the B operand of the next layer's product over the same 16 rows. Products
// over 64 features use gfx950's 16x16x32 BF16 instruction (two per 16
// output rows instead of four), whose lane l holds k = 8g..8g+7: its B
// operand for features [32t, 32t + 32) is the pair of accumulator tiles 2t
// and 2t + 1 side by side (features 32t + 4g + v, then 32t + 16 + 4g + v),
// and its A operand takes the weight columns in that same order (two runs of
// four from LDS). The sum runs over the same features in another order.
#include "mlp.h"

#include <hip/hip_ext.h>

#include <math.h>
#include <type_traits>

namespace b2mlp {
namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;           // wavefronts per workgroup
constexpr int kMaxGradBlocks = 256; // workgroups of one gradient launch at most
constexpr int kThreads = 64 * kWaves;
constexpr int kBiasCount = 3 * kHidden + kOutPad;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ inline f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// Two 4-element halves side by side as an 8-element operand.
__device__ inline bf16x8 join8(bf16x4 lo, bf16x4 hi) {
    const short s[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    bf16x8 r;
    __builtin_memcpy(&r, s, sizeof(r));
    return r;
}

// 16x16x32: features [32t, 32t + 32) of a 64-feature product, as above.
__device__ inline f32x4 mfma32(bf16x4 aLo, bf16x4 aHi, bf16x4 bLo, bf16x4 bHi, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(join8(aLo, aHi), join8(bLo, bHi), c, 0, 0, 0);
}

// Round to nearest even BF16 by the hardware conversion (the toBf16 rule for
// finite inputs).
__device__ inline bf16x4 pack4(float a, float b, float c, float d) {
    const __bf16 h[4] = {(__bf16)a, (__bf16)b, (__bf16)c, (__bf16)d};
    bf16x4 r;
    __builtin_memcpy(&r, h, sizeof(r));
    return r;
}

// Four consecutive BF16 values (8-byte aligned) from LDS.
__device__ inline bf16x4 frag(const uint16_t* p) {
    bf16x4 r;
    __builtin_memcpy(&r, p, sizeof(r));
    return r;
}

// GELU with the Gaussian CDF, 0.5 x (1 + erf(x / sqrt 2)), and its
// derivative cdf(x) + x pdf(x). erf is Abramowitz and Stegun's rational
// approximation 7.1.26 (Handbook of Mathematical Functions, 1964; absolute
// error below 1.5e-7, far under the BF16 rounding of the activations), whose
// exponential exp(-z^2) at z = x / sqrt 2 is also the density's exp(-x^2 / 2),
// so both come from one hardware exponential and one reciprocal instead of
// the library's erff and expf.
struct Cdf {
    float cdf, pdf;
};
__device__ inline Cdf gaussCdf(float x) {
    const float z = fabsf(x) * 0.70710678118654752f;
    const float e = __expf(-0.5f * x * x);
    const float t = __builtin_amdgcn_rcpf(1.0f + 0.3275911f * z);
    const float poly =
        t * (0.254829592f + t * (-0.284496736f + t * (1.421413741f + t * (-1.453152027f + t * 1.061405429f))));
    const float erfAbs = 1.0f - poly * e;
    Cdf r;
    r.cdf = 0.5f * (1.0f + (x < 0.0f ? -erfAbs : erfAbs));
    r.pdf = 0.39894228040143268f * e;
    return r;
}
// The value, and the derivative for the backward pass: one exponential and one
// reciprocal for both.
__device__ inline float gelu(float x, float& grad) {
    const Cdf c = gaussCdf(x);
    grad = c.cdf + x * c.pdf;
    return x * c.cdf;
}

// The weights in LDS. A wavefront reads 8 bytes of four neighbouring places in
// each of 16 rows at once: with rows of 64 entries, 32 banks, eight of the rows
// meet in the same banks; 72 entries spread the 16 rows over all 64 banks.
constexpr int kLd = kHidden + 8;  // row stride of the 64-column matrices
constexpr int sW1 = 0;
constexpr int sW2 = sW1 + kHidden * kIn;
constexpr int sW3 = sW2 + kHidden * kLd;
constexpr int sW4 = sW3 + kHidden * kLd;
constexpr int sW2t = sW4 + kOutPad * kLd;
constexpr int sW3t = sW2t + kHidden * kLd;
constexpr int sW4t = sW3t + kHidden * kLd;
constexpr int sTotal = sW4t + kHidden * kOutPad;
static_assert(hW2 == hW1 + kHidden * kIn && hW4t == hW2 + (4 * kHidden + kOutPad) * kHidden,
              "the 64-column matrices lie between the two 16-column ones");

struct Smem {
    alignas(16) uint16_t w[sTotal];
    float b[kBiasCount];   // b1 | b2 | b3 | b4 (padded)
    float norm[kNorm];
};

__device__ inline void loadSmem(Smem& S, const uint16_t* wh, const float* params, const float* norm) {
    static_assert(hTotal % 8 == 0, "16-byte copies");
    const uint4* src = (const uint4*)wh;
#pragma unroll 5
    for (int i = threadIdx.x; i < hTotal / 8; i += blockDim.x) {
        const int e = 8 * i, row = (e - hW2) / kHidden;
        const int at = e < hW2 ? e : e < hW4t ? sW2 + row * kLd + (e - hW2) % kHidden : sW4t + e - hW4t;
        *(uint4*)&S.w[at] = src[i];
    }
    for (int i = threadIdx.x; i < kHidden; i += blockDim.x) {
        S.b[i] = params[kB1 + i];
        S.b[kHidden + i] = params[kB2 + i];
        S.b[2 * kHidden + i] = params[kB3 + i];
    }
    for (int i = threadIdx.x; i < kOutPad; i += blockDim.x) S.b[3 * kHidden + i] = params[kB4 + i];
    for (int i = threadIdx.x; i < kNorm; i += blockDim.x) S.norm[i] = norm[i];
}

// Input fragment of a sample (v its features 4g..4g+3), standardised; zero when
// the sample is out of range.
__device__ inline bf16x4 inputFrag(const Smem& S, const float4& v, bool valid, int g) {
    if (!valid) return pack4(0.0f, 0.0f, 0.0f, 0.0f);
    const int f = 4 * g;
    return pack4((v.x - S.norm[kNormXMean + f]) * S.norm[kNormXInv + f],
                 (v.y - S.norm[kNormXMean + f + 1]) * S.norm[kNormXInv + f + 1],
                 (v.z - S.norm[kNormXMean + f + 2]) * S.norm[kNormXInv + f + 2],
                 (v.w - S.norm[kNormXMean + f + 3]) * S.norm[kNormXInv + f + 3]);
}

__device__ inline f32x4 biasTile(const Smem& S, int base, int g) {
    f32x4 r;
    for (int j = 0; j < 4; ++j) r[j] = S.b[base + 4 * g + j];
    return r;
}

// The product of weight rows [16mt, 16mt + 16) (row stride ldw, in LDS at
// wOff) with the four 16-feature tiles in[0..3] of a 64-feature input, added
// to acc: two 16x16x32 products.
__device__ inline f32x4 product64(const Smem& S, int wOff, int ldw, int mt, const bf16x4* in, f32x4 acc, int g,
                                  int c) {
    const uint16_t* row = &S.w[wOff + (16 * mt + c) * ldw];
#pragma unroll
    for (int t = 0; t < 2; ++t)
        acc = mfma32(frag(row + 32 * t + 4 * g), frag(row + 32 * t + 16 + 4 * g), in[2 * t], in[2 * t + 1], acc);
    return acc;
}

// Hidden layer: W[16mt + c][.] x in + bias, its GELU in a and the GELU's
// derivative in dz; the 16-feature input layer with one 16x16x16 product, the
// 64-feature ones with product64.
template <int KT>
__device__ inline void hiddenLayer(const Smem& S, int wOff, int ldw, int bOff, const bf16x4* in, f32x4* dz,
                                   bf16x4* a, int g, int c) {
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
        f32x4 acc = biasTile(S, bOff + 16 * mt, g);
        if (KT == 1) acc = mfma(frag(&S.w[wOff + (16 * mt + c) * ldw + 4 * g]), in[0], acc);
        else acc = product64(S, wOff, ldw, mt, in, acc, g, c);
        float d[4], v[4];
        for (int j = 0; j < 4; ++j) v[j] = gelu(acc[j], d[j]);
        for (int j = 0; j < 4; ++j) dz[mt][j] = d[j];
        a[mt] = pack4(v[0], v[1], v[2], v[3]);
    }
}

__device__ inline f32x4 outputLayer(const Smem& S, const bf16x4* a3, int g, int c) {
    return product64(S, sW4, kLd, 0, a3, biasTile(S, 3 * kHidden, g), g, c);
}

// ------------------------------------------------------------ inference
// MODE 0: y[2s], y[2s+1] = outputs (raw units).
// MODE 1: impulses of fresh contact points (see mlpPredictImpulses).
// MODE 2: impulses of any contact point as the carried impulse (features 9
//         and 15, velocity-change units) plus the outputs.
template <int MODE>
__global__ __launch_bounds__(kThreads) void k_mlp_infer(const uint16_t* wh, const float* params, const float* norm,
                                                        const float* x, int count, const int* countDev, float* y,
                                                        const int* ref, const float4* nf, float4* imp) {
    __shared__ Smem S;
    loadSmem(S, wh, params, norm);
    __syncthreads();
    const int n = countDev ? min(*countDev, count) : count;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane >> 4, c = lane & 15;
    const int tiles = (n + 15) / 16;
    for (int t = blockIdx.x * kWaves + wave; t < tiles; t += gridDim.x * kWaves) {
        const long long s = (long long)t * 16 + c;
        const bool valid = s < n;
        const float4 xv = valid ? *(const float4*)(x + s * kIn + 4 * g) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        bf16x4 x0[1] = {inputFrag(S, xv, valid, g)};
        f32x4 z[4];
        bf16x4 a1[4], a2[4], a3[4];
        hiddenLayer<1>(S, sW1, kIn, 0, x0, z, a1, g, c);
        hiddenLayer<4>(S, sW2, kLd, kHidden, a1, z, a2, g, c);
        hiddenLayer<4>(S, sW3, kLd, 2 * kHidden, a2, z, a3, g, c);
        const f32x4 o = outputLayer(S, a3, g, c);
        if (g == 0 && valid) {
            const float y0 = o[0] * S.norm[kNormYStd] + S.norm[kNormYMean];
            const float y1 = o[1] * S.norm[kNormYStd + 1] + S.norm[kNormYMean + 1];
            if (MODE == 0) {
                y[2 * s] = y0;
                y[2 * s + 1] = y1;
            } else {
                // outputs are in velocity-change units: scale by the
                // point's normal and tangent mass (features 10, 11)
                const int r = ref[s];
                const int k = r >> 1, j = r & 1;
                const float mu = nf[k].z;
                const float un = MODE == 2 ? y0 + x[s * kIn + 9] : y0;
                const float ut = MODE == 2 ? y1 + x[s * kIn + 15] : y1;
                const float yn = un * x[s * kIn + 10], yt = ut * x[s * kIn + 11];
                const float ln = yn > 0.0f ? yn : 0.0f;
                const float lim = mu * ln;
                const float lt = yt < -lim ? -lim : (yt > lim ? lim : yt);
                float* p = (float*)&imp[k];
                p[2 * j] = ln;
                p[2 * j + 1] = lt;
            }
        }
    }
}

// ------------------------------------------------------------ training
// Per-wave 16x16 transpose through LDS: in holds rows 4g..4g+3 of column c;
// the result holds row c, columns 4g..4g+3, as BF16, whatever its values. For
// the output layer's gradient, and for every tile of a wavefront that met a
// value that is not finite (see k_mlp_grad).
__device__ inline bf16x4 transposeF(float (*T)[17], f32x4 d, int g, int c) {
    for (int j = 0; j < 4; ++j) T[4 * g + j][c] = d[j];
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const bf16x4 r = pack4(T[c][4 * g], T[c][4 * g + 1], T[c][4 * g + 2], T[c][4 * g + 3]);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    return r;
}
__device__ inline bf16x4 packTile(f32x4 d) { return pack4(d[0], d[1], d[2], d[3]); }

// The same transpose on the matrix cores: read as an A operand, rows 4g..4g+3
// of column c are the transposed matrix, and its product with the identity
// has it in the accumulator's layout. Every sum is one value and zeros, so
// nothing is rounded as long as all values are finite (an infinite one times
// the identity's zeros is a NaN in its whole row); 25 of them a tile are 25
// products instead of 25 trips to LDS of four writes and four reads.
__device__ inline bf16x4 identityTile(int g, int c) {
    return pack4(4 * g == c ? 1.0f : 0.0f, 4 * g + 1 == c ? 1.0f : 0.0f, 4 * g + 2 == c ? 1.0f : 0.0f,
                 4 * g + 3 == c ? 1.0f : 0.0f);
}
template <bool kFinite>
__device__ inline bf16x4 transpose(bf16x4 d, bf16x4 identity, float (*T)[17], int g, int c) {
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (kFinite) return packTile(mfma(d, identity, zero));
    f32x4 v;
    for (int j = 0; j < 4; ++j) v[j] = __uint_as_float((uint32_t)(uint16_t)d[j] << 16);
    return transposeF(T, v, g, c);
}

// Sum over the 16 lanes that share g (lanes 16g..16g+15): neighbours, pairs,
// then the mirrored halves, in data-parallel moves instead of trips to LDS.
template <int kMove>
__device__ inline float moved(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kMove, 0xF, 0xF, true));
}
__device__ inline float groupSum16(float v) {
    v += moved<0xB1>(v);   // lanes 1, 0, 3, 2
    v += moved<0x4E>(v);   // lanes 2, 3, 0, 1
    v += moved<0x141>(v);  // half rows mirrored
    v += moved<0x140>(v);  // rows mirrored
    return v;
}

// A workgroup's sums in LDS: like the parameter vector, with row strides at
// which the four rows that a wavefront adds to at once are 16 banks apart.
constexpr int kRedIn = kIn + 4, kRedLd = kHidden + 4;
constexpr int rB1 = kHidden * kRedIn;
constexpr int rW2 = rB1 + kHidden;
constexpr int rB2 = rW2 + kHidden * kRedLd;
constexpr int rW3 = rB2 + kHidden;
constexpr int rB3 = rW3 + kHidden * kRedLd;
constexpr int rW4 = rB3 + kHidden;
constexpr int rB4 = rW4 + kOutPad * kRedLd;
constexpr int rTotal = rB4 + kOutPad;
__device__ inline int redAt(int i) {
    auto row = [](int j, int width, int ld) { return j / width * ld + j % width; };
    if (i < kB1) return row(i, kIn, kRedIn);
    if (i < kW2) return rB1 + i - kB1;
    if (i < kB2) return rW2 + row(i - kW2, kHidden, kRedLd);
    if (i < kW3) return rB2 + i - kB2;
    if (i < kB3) return rW3 + row(i - kW3, kHidden, kRedLd);
    if (i < kW4) return rB3 + i - kB3;
    if (i < kB4) return rW4 + row(i - kW4, kHidden, kRedLd);
    return rB4 + i - kB4;
}

// Bound by its one wavefront per SIMD (its sums are half the registers): the
// instructions of a tile one after another, and by what it does once: of 58 us
// for 65536 samples, four tiles a wavefront, the tiles take about 40 us and the
// sums' reduction most of the rest. 89 us with transposes through LDS, the
// GELU's exponential computed again for its derivative and one wavefront
// reducing at a time. Every sum keeps one order, wavefront after wavefront: 52 us
// without, but training then rounds otherwise (and that 63 us with rows of 64
// entries in LDS).
__global__ __launch_bounds__(kThreads) void k_mlp_grad(const uint16_t* wh, const float* params, const float* norm,
                                                       const float* x, const float* tgt, const int* order, int first,
                                                       int count, float invN, float* partial) {
    __shared__ Smem S;
    __shared__ float red[rTotal];
    __shared__ float lossShared;
    __shared__ float tf[kWaves][16][17];
    loadSmem(S, wh, params, norm);
    if (threadIdx.x == 0) lossShared = 0.0f;
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = lane >> 4, c = lane & 15;
    float (*TF)[17] = tf[wave];
    const bf16x4 ident = identityTile(g, c);

    f32x4 gW1[4], gW2[4][4], gW3[4][4], gW4[4];
    float gb1[4][4], gb2[4][4], gb3[4][4], gb4[4];
    const f32x4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    float loss = 0.0f;
    auto sums = [&](auto finite) {
        constexpr bool kFinite = decltype(finite)::value;
        for (int i = 0; i < 4; ++i) {
            gW1[i] = zero4;
            gW4[i] = zero4;
            gb4[i] = 0.0f;
            for (int k = 0; k < 4; ++k) {
                gW2[i][k] = zero4;
                gW3[i][k] = zero4;
                gb1[i][k] = gb2[i][k] = gb3[i][k] = 0.0f;
            }
        }
        loss = 0.0f;
        const int tiles = (count + 15) / 16;
        for (int t = blockIdx.x * kWaves + wave; t < tiles; t += gridDim.x * kWaves) {
            const long long local = (long long)t * 16 + c;
            const bool valid = local < count;
            const long long s = valid ? (order ? (long long)order[first + local] : first + local) : 0;
            const float4 xv = *(const float4*)(x + s * kIn + 4 * g);
            const float2 tv = *(const float2*)(tgt + 2 * s);
            // forward, keeping activations and their derivatives
            bf16x4 x0[1] = {inputFrag(S, xv, valid, g)};
            f32x4 z1[4], z2[4], z3[4];  // the GELUs' derivatives
            bf16x4 a1[4], a2[4], a3[4];
            hiddenLayer<1>(S, sW1, kIn, 0, x0, z1, a1, g, c);
            hiddenLayer<4>(S, sW2, kLd, kHidden, a1, z2, a2, g, c);
            hiddenLayer<4>(S, sW3, kLd, 2 * kHidden, a2, z3, a3, g, c);
            const f32x4 o = outputLayer(S, a3, g, c);
            // dL/dy on standardised targets (rows 0, 1 of the output tile are in lanes g == 0)
            f32x4 d4 = zero4;
            if (g == 0 && valid) {
                const float t0 = (tv.x - S.norm[kNormYMean]) / S.norm[kNormYStd];
                const float t1 = (tv.y - S.norm[kNormYMean + 1]) / S.norm[kNormYStd + 1];
                const float e0 = o[0] - t0, e1 = o[1] - t1;
                loss += 0.5f * (e0 * e0 + e1 * e1) * invN;
                d4[0] = e0 * invN;
                d4[1] = e1 * invN;
            }
            // layer 4: weight gradient and backward-data
            {
                const bf16x4 dT = transposeF(TF, d4, g, c);
    #pragma unroll
                for (int ni = 0; ni < 4; ++ni) gW4[ni] = mfma(dT, transpose<kFinite>(a3[ni], ident, TF, g, c), gW4[ni]);
                for (int j = 0; j < 4; ++j) gb4[j] += d4[j];
            }
            f32x4 d3[4];
            {
                const bf16x4 dB = packTile(d4);
    #pragma unroll
                for (int mt = 0; mt < 4; ++mt) {
                    f32x4 acc = mfma(frag(&S.w[sW4t + (16 * mt + c) * kOutPad + 4 * g]), dB, zero4);
                    for (int j = 0; j < 4; ++j) acc[j] *= z3[mt][j];
                    d3[mt] = acc;
                }
            }
            // layer 3
            {
                bf16x4 hT[4], dB[4];
                for (int ni = 0; ni < 4; ++ni) hT[ni] = transpose<kFinite>(a2[ni], ident, TF, g, c);
    #pragma unroll
                for (int mo = 0; mo < 4; ++mo) {
                    dB[mo] = packTile(d3[mo]);
                    const bf16x4 dT = transpose<kFinite>(dB[mo], ident, TF, g, c);
    #pragma unroll
                    for (int ni = 0; ni < 4; ++ni) gW3[mo][ni] = mfma(dT, hT[ni], gW3[mo][ni]);
                    for (int j = 0; j < 4; ++j) gb3[mo][j] += d3[mo][j];
                }
                f32x4 d2[4];
    #pragma unroll
                for (int mt = 0; mt < 4; ++mt) {
                    f32x4 acc = product64(S, sW3t, kLd, mt, dB, zero4, g, c);
                    for (int j = 0; j < 4; ++j) acc[j] *= z2[mt][j];
                    d2[mt] = acc;
                }
                // layer 2
                for (int ni = 0; ni < 4; ++ni) hT[ni] = transpose<kFinite>(a1[ni], ident, TF, g, c);
    #pragma unroll
                for (int mo = 0; mo < 4; ++mo) {
                    dB[mo] = packTile(d2[mo]);
                    const bf16x4 dT = transpose<kFinite>(dB[mo], ident, TF, g, c);
    #pragma unroll
                    for (int ni = 0; ni < 4; ++ni) gW2[mo][ni] = mfma(dT, hT[ni], gW2[mo][ni]);
                    for (int j = 0; j < 4; ++j) gb2[mo][j] += d2[mo][j];
                }
                // layer 1
                const bf16x4 xT = transpose<kFinite>(x0[0], ident, TF, g, c);
    #pragma unroll
                for (int mt = 0; mt < 4; ++mt) {
                    f32x4 acc = product64(S, sW2t, kLd, mt, dB, zero4, g, c);
                    for (int j = 0; j < 4; ++j) acc[j] *= z1[mt][j];
                    const bf16x4 dT = transpose<kFinite>(packTile(acc), ident, TF, g, c);
                    gW1[mt] = mfma(dT, xT, gW1[mt]);
                    for (int j = 0; j < 4; ++j) gb1[mt][j] += acc[j];
                }
            }
        }
    };
    sums(std::true_type{});
    // A tile with a value that is not finite leaves one in every sum it is part
    // of (infinity times anything is infinite or NaN), so finite sums prove the
    // transposes exact. Otherwise the wavefront's tiles are summed again with
    // transposes that keep each value in its place. (The test costs 0.3 us of
    // the kernel's 57 us.)
    float probe = 0.0f;
    for (int i = 0; i < 4; ++i)
        for (int j = 0; j < 4; ++j) {
            probe += 0.0f * gW1[i][j] + 0.0f * gW4[i][j];
            for (int k = 0; k < 4; ++k) probe += 0.0f * gW2[i][k][j] + 0.0f * gW3[i][k][j];
        }
    if (__any(!(probe == 0.0f))) sums(std::false_type{});
    // Reduce the four wavefronts in LDS, each entry in wavefront order: the sums
    // are added by quarters, a wavefront one turn behind the one before it, so
    // that four work at once (each lane owns distinct entries, so plain
    // read-add-writes, the first wavefront's a write): accumulator element j of tile (mo, ni) is
    // dW[16mo + 4g + j][16ni + c]. Then the workgroup's sums go to its row of
    // `partial`, which k_mlp_reduce adds up in a fixed order: the gradient does
    // not depend on the schedule.
    float l = loss;
    for (int off = 1; off < 64; off <<= 1) l += __shfl_xor(l, off);
#pragma clang loop unroll(disable)
    for (int turn = 0; turn < kWaves + 3; ++turn) {
        auto add = [&](int i, float v) { red[i] = (wave == 0 ? 0.0f : red[i]) + v; };
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (turn - wave != q) continue;
            for (int j = 0; j < 4; ++j) {
                const int o = 16 * q + 4 * g + j;
                add(o * kRedIn + c, gW1[q][j]);
                for (int ni = 0; ni < 4; ++ni) {
                    add(rW2 + o * kRedLd + 16 * ni + c, gW2[q][ni][j]);
                    add(rW3 + o * kRedLd + 16 * ni + c, gW3[q][ni][j]);
                }
                add(rW4 + (4 * g + j) * kRedLd + 16 * q + c, gW4[q][j]);
                const float s1 = groupSum16(gb1[q][j]), s2 = groupSum16(gb2[q][j]), s3 = groupSum16(gb3[q][j]);
                if (c == 0) {
                    add(rB1 + o, s1);
                    add(rB2 + o, s2);
                    add(rB3 + o, s3);
                }
            }
            if (q == 0)
                for (int j = 0; j < 4; ++j) {
                    const float s4 = groupSum16(gb4[j]);
                    if (c == 0) add(rB4 + 4 * g + j, s4);
                }
        }
        if (lane == 0 && wave == turn) lossShared += l;
        __syncthreads();
    }
    float* row = partial + (size_t)blockIdx.x * (kParams + 1);
    for (int i = threadIdx.x; i < kParams; i += blockDim.x) row[i] = red[redAt(i)];
    if (threadIdx.x == 0) row[kParams] = lossShared;
}

// BF16 image entries of parameter i (weights only; biases stay FP32).
__device__ inline void writeImage(uint16_t* wh, int i, float v) {
    const uint16_t h = toBf16(v);
    if (i < kB1) {
        wh[hW1 + i] = h;
    } else if (i >= kW2 && i < kB2) {
        const int r = i - kW2, o = r / kHidden, in = r % kHidden;
        wh[hW2 + r] = h;
        wh[hW2t + in * kHidden + o] = h;
    } else if (i >= kW3 && i < kB3) {
        const int r = i - kW3, o = r / kHidden, in = r % kHidden;
        wh[hW3 + r] = h;
        wh[hW3t + in * kHidden + o] = h;
    } else if (i >= kW4 && i < kB4) {
        const int r = i - kW4, o = r / kHidden, in = r % kHidden;
        wh[hW4 + r] = h;
        wh[hW4t + in * kOutPad + o] = h;
    }
}

__global__ void k_mlp_image(const float* params, uint16_t* wh) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kParams) writeImage(wh, i, params[i]);
}

struct AdamState {
    float *params, *m, *v;
    uint16_t* wh;
    float lr, c1, c2;
};
__device__ inline void adamOne(const AdamState& a, int i, float gi) {
    const float mi = 0.9f * a.m[i] + 0.1f * gi;
    const float vi = 0.999f * a.v[i] + 0.001f * gi * gi;
    a.m[i] = mi;
    a.v[i] = vi;
    const float p = a.params[i] - a.lr * (mi * a.c1) / (sqrtf(vi * a.c2) + 1e-8f);
    a.params[i] = p;
    writeImage(a.wh, i, p);
}

// Sum of the workgroups' rows added to the gradient and the loss, in a
// fixed order: a workgroup takes kReduceCols consecutive entries; its
// kReduceSplit lane groups each sum every kReduceSplit-th row in row order
// (coalesced across the entries), then the groups' sums are added in group
// order. In training the entries' Adam step follows in the same lanes.
// Bound by the trips for the rows (10.7 MB at 256 rows): 18 us with a load at
// a time, 5.1 us with 16 in flight and the Adam step, which took 4.9 us as a
// launch of its own.
constexpr int kReduceCols = 64, kReduceSplit = 4;
template <bool kAdam>
__global__ __launch_bounds__(kReduceCols * kReduceSplit) void k_mlp_reduce(const float* partial, int rows,
                                                                            float* grad, float* loss, AdamState adam) {
    __shared__ float part[kReduceSplit][kReduceCols];
    const int col = threadIdx.x % kReduceCols, grp = threadIdx.x / kReduceCols;
    const int i = blockIdx.x * kReduceCols + col;
    float acc = 0.0f;
    if (i <= kParams) {
#pragma unroll 16
        for (int r = grp; r < rows; r += kReduceSplit) acc += partial[(size_t)r * (kParams + 1) + i];
    }
    part[grp][col] = acc;
    __syncthreads();
    if (grp != 0 || i > kParams) return;
    float sum = part[0][col];
#pragma unroll
    for (int k = 1; k < kReduceSplit; ++k) sum += part[k][col];
    if (i == kParams) {
        *loss += sum;
    } else if (kAdam) {
        adamOne(adam, i, grad[i] + sum);
        grad[i] = 0.0f;
    } else {
        grad[i] += sum;
    }
}

int gridFor(int count) {
    const int tiles = (count + 15) / 16;
    int g = (tiles + kWaves - 1) / kWaves;
    if (g < 1) g = 1;
    return g < 1024 ? g : 1024;
}

}  // namespace

hipError_t mlpAlloc(Net& n, hipStream_t s) {
    hipError_t e;
    if ((e = hipMalloc((void**)&n.params, sizeof(float) * kParams)) != hipSuccess) return e;
    if ((e = hipMalloc((void**)&n.grad, sizeof(float) * kParams)) != hipSuccess) return e;
    if ((e = hipMalloc((void**)&n.m, sizeof(float) * kParams)) != hipSuccess) return e;
    if ((e = hipMalloc((void**)&n.v, sizeof(float) * kParams)) != hipSuccess) return e;
    if ((e = hipMalloc((void**)&n.wh, sizeof(uint16_t) * hTotal)) != hipSuccess) return e;
    if ((e = hipMalloc((void**)&n.norm, sizeof(float) * kNorm)) != hipSuccess) return e;
    if ((e = hipMalloc((void**)&n.loss, sizeof(float))) != hipSuccess) return e;
    if ((e = hipMalloc((void**)&n.partial, sizeof(float) * kMaxGradBlocks * (kParams + 1))) != hipSuccess) return e;
    if ((e = hipMemsetAsync(n.params, 0, sizeof(float) * kParams, s)) != hipSuccess) return e;
    if ((e = hipMemsetAsync(n.grad, 0, sizeof(float) * kParams, s)) != hipSuccess) return e;
    if ((e = hipMemsetAsync(n.m, 0, sizeof(float) * kParams, s)) != hipSuccess) return e;
    if ((e = hipMemsetAsync(n.v, 0, sizeof(float) * kParams, s)) != hipSuccess) return e;
    if ((e = hipMemsetAsync(n.wh, 0, sizeof(uint16_t) * hTotal, s)) != hipSuccess) return e;
    if ((e = hipMemsetAsync(n.norm, 0, sizeof(float) * kNorm, s)) != hipSuccess) return e;
    return hipMemsetAsync(n.loss, 0, sizeof(float), s);
}

void mlpFree(Net& n) {
    void* ps[] = {n.params, n.grad, n.m, n.v, n.wh, n.norm, n.loss, n.partial};
    for (void* p : ps)
        if (p) (void)hipFree(p);
    n = Net();
}

hipError_t mlpPrepare(const Net& n, hipStream_t s) {
    hipLaunchKernelGGL(k_mlp_image, dim3((kParams + 255) / 256), dim3(256), 0, s, n.params, n.wh);
    return hipGetLastError();
}

hipError_t mlpForward(const Net& n, const float* x, int count, float* y, hipStream_t s, hipEvent_t e0,
                      hipEvent_t e1) {
    if (count <= 0) return hipSuccess;
    hipExtLaunchKernelGGL(k_mlp_infer<0>, dim3(gridFor(count)), dim3(kThreads), 0, s, e0, e1, 0, n.wh, n.params,
                          n.norm, x, count, (const int*)nullptr, y, (const int*)nullptr, (const float4*)nullptr,
                          (float4*)nullptr);
    return hipGetLastError();
}

hipError_t mlpPredictImpulses(const Net& n, const float* feat, const int* ref, const int* countDev, int maxCount,
                              const float4* normalFriction, float4* imp, bool delta, hipStream_t s, hipEvent_t e0,
                              hipEvent_t e1) {
    if (maxCount <= 0) return hipSuccess;
    if (delta)
        hipExtLaunchKernelGGL(k_mlp_infer<2>, dim3(gridFor(maxCount)), dim3(kThreads), 0, s, e0, e1, 0, n.wh,
                              n.params, n.norm, feat, maxCount, countDev, (float*)nullptr, ref, normalFriction, imp);
    else
        hipExtLaunchKernelGGL(k_mlp_infer<1>, dim3(gridFor(maxCount)), dim3(kThreads), 0, s, e0, e1, 0, n.wh,
                              n.params, n.norm, feat, maxCount, countDev, (float*)nullptr, ref, normalFriction, imp);
    return hipGetLastError();
}

namespace {
int launchGrad(const Net& n, const float* x, const float* t, const int* order, int first, int count, hipStream_t s,
               hipEvent_t e0, hipEvent_t e1) {
    // one workgroup per CU at most (the kernel's LDS allows one), each
    // wavefront taking as many 16-sample tiles as needed
    const int tiles = (count + 15) / 16;
    int grid = (tiles + kWaves - 1) / kWaves;
    if (grid > kMaxGradBlocks) grid = kMaxGradBlocks;
    if (grid < 1) grid = 1;
    hipExtLaunchKernelGGL(k_mlp_grad, dim3(grid), dim3(kThreads), 0, s, e0, e1, 0, n.wh, n.params, n.norm, x, t,
                          order, first, count, 1.0f / (float)count, n.partial);
    return grid;
}
constexpr int kReduceGrid = (kParams + 1 + kReduceCols - 1) / kReduceCols;
}  // namespace

hipError_t mlpGradient(const Net& n, const float* x, const float* t, const int* order, int first, int count,
                       hipStream_t s, hipEvent_t e0, hipEvent_t e1) {
    if (count <= 0) return hipSuccess;
    const int grid = launchGrad(n, x, t, order, first, count, s, e0, e1);
    hipLaunchKernelGGL(k_mlp_reduce<false>, dim3(kReduceGrid), dim3(kReduceCols * kReduceSplit), 0, s, n.partial, grid,
                       n.grad, n.loss, AdamState{});
    return hipGetLastError();
}

hipError_t mlpTrainStep(Net& n, const float* x, const float* t, const int* order, int first, int count, float lr,
                        hipStream_t s, hipEvent_t e0, hipEvent_t e1) {
    if (count <= 0) return hipSuccess;
    const int grid = launchGrad(n, x, t, order, first, count, s, e0, e1);
    ++n.adamStep;
    const double c1 = 1.0 / (1.0 - pow(0.9, n.adamStep));
    const double c2 = 1.0 / (1.0 - pow(0.999, n.adamStep));
    const AdamState adam{n.params, n.m, n.v, n.wh, lr, (float)c1, (float)c2};
    hipLaunchKernelGGL(k_mlp_reduce<true>, dim3(kReduceGrid), dim3(kReduceCols * kReduceSplit), 0, s, n.partial, grid,
                       n.grad, n.loss, adam);
    return hipGetLastError();
}

}  // namespace b2mlp
