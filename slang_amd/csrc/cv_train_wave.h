// cv_train_wave.h -- the training step of a network of float, every wave by itself.
//
// The step of cv_train_round.h for float networks small enough that one wave can hold all of dW in registers: up to 64-wide
// hidden layers with up to 36 tiles of 16 x 16 gradients (144 registers).  A wave takes 16 samples through forward, loss,
// backward and the dW products, with no other wave to wait for: the waves of a workgroup share the weights in LDS and meet
// only to add up their gradients at the end.  (The same networks with the samples of a round and the dW tiles spread over
// eight waves, which meet at nine barriers per 64 samples: 32-64-64-8 over 2^20 samples 462 us, layer by layer over memory
// 1558 us; here 390 us.)
//
// Layout.  v_mfma_f32_16x16x4_f32 leaves rows 4g .. 4g+3 of a 16-row tile in lane group g's four accumulator registers,
// which is the B operand of four such instructions whose k axis is those rows: a layer's accumulators are the next layer's
// operands as they lie (forward and dX = W^T dZ alike).  Only dW = sum_s dZ (x) X needs the sample index on the k axis: X
// and dZ of the wave's 16 samples also go to LDS, [sample][feature], and come back by columns; dZ_l takes the place of X_l.
// One copy of W serves both directions, by rows forward, by columns for dX.
//
// What bounds it: the matrix pipeline (32 cycles per instruction; 304 of them for 16 samples of 32-64-64-8, which keep it busy
// 65 % of the time).  Of the instantiations one spills: three layers with 33 to 64 inputs keep 136 bytes a lane in scratch memory
// (64-64-64-9 over 2^19 samples: 245 us, 32-64-64-8: 213 us).
#pragma once
#include "cv_train_round.h"

namespace cv {
namespace {

constexpr int kWaveMaxTiles = 36;

// HT: 16-unit tiles of every hidden layer (narrower ones are padded with zero weights), IT: of the input, NL layers
template <int HT_, int NL_, int IT_>
struct WaveNet {
    static constexpr int HT = HT_, NL = NL_, IT = IT_;
    static constexpr int outTiles(int l) { return l + 1 < NL ? HT : 1; }
    static constexpr int inTiles(int l) { return l == 0 ? IT : HT; }
    static constexpr uint32_t xStride(int l) { return (uint32_t)(l < NL ? inTiles(l) : 1) * 64u + 16u; }      // X_l; l == NL: dZ of the last layer
    static constexpr uint32_t wStride(int l) { return xStride(l); }
    static constexpr uint32_t wOff(int l)
    {
        uint32_t b = 0;
        for (int i = 0; i < l; ++i) b += (uint32_t)outTiles(i) * 16u * wStride(i);
        return b;
    }
    static constexpr uint32_t biasOff(int l)
    {
        uint32_t b = wOff(NL);
        for (int i = 0; i < l; ++i) b += (uint32_t)outTiles(i) * 64u;
        return b;
    }
    static constexpr uint32_t waveOff = biasOff(NL);      // the waves' vectors
    static constexpr uint32_t xOff(int l)
    {
        uint32_t b = 0;
        for (int i = 0; i < l; ++i) b += 16u * xStride(i);
        return b;
    }
    static constexpr uint32_t waveBytes = xOff(NL + 1);
    static constexpr uint32_t ldsBytes = waveOff + 8u * waveBytes + 16u;
    static constexpr int tileBase(int l)
    {
        int b = 0;
        for (int i = 0; i < l; ++i) b += outTiles(i) * inTiles(i);
        return b;
    }
    static constexpr int tiles = tileBase(NL);
    static constexpr int rowBase(int l) { return l * HT; }
    static constexpr int rows = rowBase(NL - 1) + 1;
    static constexpr bool fits = tiles <= kWaveMaxTiles && ldsBytes <= 160u * 1024u;
};

// The lanes of a wave exchange vectors through LDS, whose accesses the hardware keeps in order: what lies before this stays
// before it for every lane.  No instruction.
__device__ __forceinline__ void orderLanes()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <class Net>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void trainWaveKernel(const RoundArgs a)
{
    typedef RoundMma<float> M;
    constexpr int NL = Net::NL, HT = Net::HT, IT = Net::IT;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    uint32_t* const ldsLossMax = (uint32_t*)(lds + Net::ldsBytes - 16u);

    for (uint32_t i = threadIdx.x; i < Net::ldsBytes / 16u; i += 512u) ((u32x4*)lds)[i] = u32x4{0u, 0u, 0u, 0u};
    __syncthreads();
    stageRoundWeights<float, NL, (IT > HT ? IT : HT)>(a.layers, lds);
    __syncthreads();

    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint8_t* const mine = lds + Net::waveOff + (uint32_t)wave * Net::waveBytes;

    floatx4 accW[Net::tiles];
    float accB[Net::rows];
#pragma unroll
    for (int i = 0; i < Net::tiles; ++i) accW[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < Net::rows; ++i) accB[i] = 0.f;
    float lossAcc = 0.f, lossMaxAcc = 0.f;

    const int in0 = a.layers[0].in, topOut = a.layers[NL - 1].out, topAct = a.layers[NL - 1].act;
    const float topSlope = a.layers[NL - 1].slope;
    const uint32_t lastSample = a.batch - 1u, numTiles = lastSample / 16u + 1u;

    // the tile's input as B operands (lane 16g + j: features 16q + 4g .. of sample j) and its targets (rows 4g .. 4g+3)
    auto fetch = [&](floatx4 (&x)[IT], float (&t)[4], uint32_t tile) {
        const uint32_t s = min(tile * 16u + n, lastSample);
        const uint8_t* row = a.in + (size_t)s * a.inStride;
        if (a.inPieces) {
#pragma unroll
            for (int q = 0; q < IT; ++q) x[q] = *(const floatx4*)(row + 16 * min(4 * q + g, a.inPieces - 1));
        } else {
#pragma unroll
            for (int q = 0; q < IT; ++q)
#pragma unroll
                for (int r = 0; r < 4; ++r) x[q][r] = *(const float*)(row + 4 * min(16 * q + 4 * g + r, in0 - 1));
        }
        if (a.targets) {
            const uint8_t* p = a.targets + (size_t)s * a.targetStride;
#pragma unroll
            for (int r = 0; r < 4; ++r) t[r] = *(const float*)(p + 4 * min(4 * g + r, topOut - 1));
        }
    };

    auto oneTile = [&](const floatx4 (&xin)[IT], const float (&tgt)[4], uint32_t tile) {
        constexpr int MAXT = IT > HT ? IT : HT;
        floatx4 x[MAXT];                     // B operands: the current layer's input, later dZ
        orderLanes();                        // (the tile before has read X and dZ)
#pragma unroll
        for (int q = 0; q < IT; ++q) {
#pragma unroll
            for (int r = 0; r < 4; ++r) x[q][r] = 16 * q + 4 * g + r < in0 ? xin[q][r] : 0.f;
            *(floatx4*)(mine + Net::xOff(0) + (uint32_t)n * Net::xStride(0) + 64 * q + 16 * g) = x[q];
        }
        float tgtAll = 0.f;
        if (!a.targets) {
            // sin(sum of the inputs), each lane group a quarter of them, as the other steps form it
            orderLanes();
            const int gs = (int)optGS((uint32_t)in0);
            const float* xs = (const float*)(mine + Net::xOff(0) + (uint32_t)n * Net::xStride(0));
            float part = 0.f;
            for (int q = 0; q < gs; ++q) part += g * gs + q < in0 ? xs[g * gs + q] : 0.f;
            tgtAll = sinf(sumOverGroups(part));
        }

        // ---- forward ----------------------------------------------------------------------------------------------------
        auto product = [&](auto lc, floatx4* acc) {
            constexpr int l = decltype(lc)::value, OT = Net::outTiles(l), KT = Net::inTiles(l);
            const uint8_t* w = lds + Net::wOff(l) + (uint32_t)n * Net::wStride(l) + 16 * g;
#pragma unroll
            for (int t = 0; t < OT; ++t) acc[t] = *(const floatx4*)(lds + Net::biasOff(l) + 64 * t + 16 * g);
#pragma unroll
            for (int q = 0; q < KT; ++q) {
                floatx4 wv[OT];
#pragma unroll
                for (int t = 0; t < OT; ++t) wv[t] = *(const floatx4*)(w + (uint32_t)(16 * t) * Net::wStride(l) + 64 * q);
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int t = 0; t < OT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[t][r], x[q][r], acc[t], 0, 0, 0);
            }
        };
        staticFor<0, NL - 1>([&](auto lc) {
            constexpr int l = decltype(lc)::value;
            floatx4 acc[HT];
            product(lc, acc);
            const int act = a.layers[l].act;
            const float slope = a.layers[l].slope;
            if (act == kActRelu) {
#pragma unroll
                for (int t = 0; t < HT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[t][r] = acc[t][r] > 0.f ? acc[t][r] : (acc[t][r] == 0.f ? 0.f : -0.f);      // (NaN: -0)
            } else if (act == kActLeakyRelu) {
#pragma unroll
                for (int t = 0; t < HT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) { const float u = acc[t][r] + 0.f; acc[t][r] = fmaxf(u, u * slope); }
            }
#pragma unroll
            for (int t = 0; t < HT; ++t) {
                x[t] = acc[t];
                *(floatx4*)(mine + Net::xOff(l + 1) + (uint32_t)n * Net::xStride(l + 1) + 64 * t + 16 * g) = acc[t];
            }
        });
        // ---- loss and its gradient at the last pre-activations -----------------------------------------------------------
        {
            floatx4 z[1];
            product(std::integral_constant<int, NL - 1>{}, z);
            const bool live = tile * 16u + n < a.batch;
            float sampleLoss = 0.f;
            floatx4 dz;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const bool on = live && 4 * g + r < topOut;
                const float v = z[0][r];
                float y = v;
                if (topAct == kActRelu) y = v > 0.f ? v : 0.f;
                if (topAct == kActLeakyRelu) y = fmaxf(v, v * topSlope);
                const float diff = y - (a.targets ? tgt[r] : tgtAll);
                sampleLoss += on ? diff * diff : 0.f;
                const float gv = 2.0f * diff * a.lossScale, hg = 0.5f * gv;
                float d = gv;
                if (topAct == kActRelu) d = v > 0.f ? gv : (v == 0.f ? hg : 0.f);
                if (topAct == kActLeakyRelu) d = v > 0.f ? gv : (v == 0.f ? hg + hg * topSlope : gv * topSlope);
                dz[r] = on ? d : 0.f;
            }
            lossAcc += sampleLoss;
            if (a.wantLossMax) {
                const float whole = sumOverGroups(sampleLoss);
                lossMaxAcc = (whole > lossMaxAcc || whole != whole) ? whole : lossMaxAcc;
            }
            x[0] = dz;
            *(floatx4*)(mine + Net::xOff(NL) + (uint32_t)n * Net::xStride(NL) + 16 * g) = dz;
        }
        orderLanes();
        // ---- backward -----------------------------------------------------------------------------------------------------
        staticFor<0, NL>([&](auto ic) {
            constexpr int l = NL - 1 - decltype(ic)::value, OT = Net::outTiles(l), NI = Net::inTiles(l);
            // dX = W^T dZ
            floatx4 gx[l > 0 ? HT : 1];
            if constexpr (l > 0) {
#pragma unroll
                for (int t = 0; t < HT; ++t) gx[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int q = 0; q < OT; ++q) {
                    floatx4 wv[HT];
#pragma unroll
                    for (int t = 0; t < HT; ++t) wv[t] = M::readColumn(lds + Net::wOff(l) + (uint32_t)(16 * q) * Net::wStride(l) + 64 * t, Net::wStride(l), g, n);
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int t = 0; t < HT; ++t) gx[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[t][r], x[q][r], gx[t], 0, 0, 0);
                }
            }
            // dW += dZ (x) X, db += dZ
            {
                floatx4 dz[OT], xv[NI];
#pragma unroll
                for (int t = 0; t < OT; ++t) dz[t] = M::readColumn(mine + Net::xOff(l + 1) + 64 * t, Net::xStride(l + 1), g, n);
#pragma unroll
                for (int u = 0; u < NI; ++u) xv[u] = M::readColumn(mine + Net::xOff(l) + 64 * u, Net::xStride(l), g, n);
#pragma unroll
                for (int t = 0; t < OT; ++t) accB[Net::rowBase(l) + t] = M::sum(dz[t], accB[Net::rowBase(l) + t]);
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int t = 0; t < OT; ++t)
#pragma unroll
                        for (int u = 0; u < NI; ++u) {
                            floatx4& w = accW[Net::tileBase(l) + t * NI + u];
                            w = __builtin_amdgcn_mfma_f32_16x16x4f32(dz[t][r], xv[u][r], w, 0, 0, 0);
                        }
            }
            // through the activation of the layer below, in the place of its output
            if constexpr (l > 0) {
                orderLanes();                // (dW has read X_l)
#pragma unroll
                for (int t = 0; t < HT; ++t) {
                    uint8_t* p = mine + Net::xOff(l) + (uint32_t)n * Net::xStride(l) + 64 * t + 16 * g;
                    x[t] = M::storeGradient(p, gx[t], a.layers[l - 1].act, a.layers[l - 1].slope);
                }
                orderLanes();
            }
        });
    };

    {
        const uint32_t stride = gridDim.x * 8u;
        uint32_t tile = blockIdx.x * 8u + wave;
        floatx4 cur[IT], nxt[IT];
        float ct[4] = {0.f, 0.f, 0.f, 0.f}, nt[4] = {0.f, 0.f, 0.f, 0.f};
        fetch(cur, ct, tile);
        for (; tile < numTiles; tile += stride) {
            fetch(nxt, nt, tile + stride);
            asm volatile("" ::: "memory");      // the requests stay above the tile ...
            oneTile(cur, ct, tile);
#pragma unroll
            for (int q = 0; q < IT; ++q) { pinHere(nxt[q]); cur[q] = nxt[q]; }      // ... and are first touched below it
#pragma unroll
            for (int r = 0; r < 4; ++r) { pinHere(nt[r]); ct[r] = nt[r]; }
        }
    }

    // ---- the workgroup's partial: eight waves added in a fixed order through LDS, some tiles at a time -----------------------
    __syncthreads();
    float* part = a.partials + (size_t)blockIdx.x * a.partialFloats;
    float* red = (float*)lds;
    if (a.wantLossMax) noteLossMax(ldsLossMax, lossMaxAcc);
    red[threadIdx.x] = lossAcc;
    __syncthreads();
    if (wave == 0) {
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < 8; ++w) s += red[64 * w + lane];
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) s += __shfl_xor(s, d, 64);
        if (lane == 0) {
            part[a.partialFloats - 16] = s;
            part[a.partialFloats - 15] = __builtin_bit_cast(float, *ldsLossMax);
        }
    }
    constexpr int kAtOnce = (int)((Net::ldsBytes - 16u) / 8192u) < 16 ? (int)((Net::ldsBytes - 16u) / 8192u) : 16;
    staticFor<0, (Net::tiles + kAtOnce - 1) / kAtOnce>([&](auto pc) {
        constexpr int first = decltype(pc)::value * kAtOnce, count = Net::tiles - first < kAtOnce ? Net::tiles - first : kAtOnce;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < count; ++i) *(floatx4*)&red[(i * 8 + wave) * 256 + 4 * lane] = accW[first + i];
        __syncthreads();
        // wave w sums tiles w, w + 8, ...
#pragma unroll
        for (int i0 = 0; i0 < count; i0 += 8) {
            const int i = i0 + wave;
            if (i >= count) continue;
            int l = 0;
#pragma unroll
            for (int k = 1; k < NL; ++k) l = first + i >= Net::tileBase(k) ? k : l;
            int base = 0, ni = IT;
#pragma unroll
            for (int k = 1; k < NL; ++k) { base = l == k ? Net::tileBase(k) : base; ni = l == k ? HT : ni; }
            const int t = (first + i - base) / ni, u = (first + i - base) % ni;
            if (t >= a.layers[l].rowTiles || u >= a.layers[l].colTiles) continue;
            floatx4 s = *(const floatx4*)&red[i * 8 * 256 + 4 * lane];
#pragma unroll
            for (int w = 1; w < 8; ++w) s += *(const floatx4*)&red[(i * 8 + w) * 256 + 4 * lane];
            const uint32_t tile = a.layers[l].tileBase + (uint32_t)(t * a.layers[l].colTiles + u);
            __builtin_nontemporal_store(s, (floatx4*)&part[tile * 256 + 4 * lane]);
        }
    });
    __syncthreads();
#pragma unroll
    for (int i = 0; i < Net::rows; ++i) {      // a row's bias gradient lies in the four lane groups
        float s = accB[i] + __shfl_xor(accB[i], 16, 64);
        s += __shfl_xor(s, 32, 64);
        if (g == 0) red[(i * 8 + wave) * 16 + n] = s;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < Net::rows * 16; e += 512) {
        const int i = e >> 4, l = i / HT < NL - 1 ? i / HT : NL - 1, t = i - Net::rowBase(l);
        if (t >= a.layers[l].rowTiles) continue;
        float s = red[i * 128 + (e & 15)];
#pragma unroll
        for (int w = 1; w < 8; ++w) s += red[(i * 8 + w) * 16 + (e & 15)];
        part[a.dwTiles * 256 + (a.layers[l].dbBase + t) * 16 + (e & 15)] = s;
    }
}

template <class Net>
hipError_t launchWave(hipStream_t stream, const TrainLaunch& t, RoundArgs& a, int numCUs)
{
    for (int l = 0; l < Net::NL; ++l) {
        a.layers[l].wOff = Net::wOff(l); a.layers[l].wStride = Net::wStride(l); a.layers[l].biasOff = Net::biasOff(l);
    }
    a.ldsBytes = Net::ldsBytes;
    const hipError_t e = allowDynamicLds<trainWaveKernel<Net>>(160 * 1024);
    if (e != hipSuccess) return e;
    const uint32_t need = (t.mlp.batch - 1u) / 128u + 1u, blocks = need < (uint32_t)numCUs ? need : (uint32_t)numCUs;
    a.finish.numPartials = blocks;
    noteKernel(false, "trainWaveKernel<f32,%d layers,inputs<=%d,hidden<=%d> + trainRoundReduceKernel", Net::NL, 16 * Net::IT, 16 * Net::HT);
    hipLaunchKernelGGL((trainWaveKernel<Net>), dim3(blocks), dim3(512), Net::ldsBytes, stream, a);
    const hipError_t e1 = hipGetLastError();
    if (e1 != hipSuccess) return e1;
    hipLaunchKernelGGL(trainRoundReduceKernel, dim3((a.partialFloats - 16u) / 64u + 1u), dim3(64 * kReduceWaves), 0, stream, a);
    return hipGetLastError();
}

} // namespace
} // namespace cv
