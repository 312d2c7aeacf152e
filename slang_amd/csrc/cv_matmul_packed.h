// cv_matmul_packed.h -- the batched matMul for vectors of any length and alignment.
//
// Vectors.  A wave takes 16 * NT samples at a time and a lane its k-slots of a sample in reads of 16 bytes at whatever element
// they begin, a tile ahead; what lies behind the end of a vector (of the next one) is cleared in registers.  Reads that would leave the
// buffer, of the last few samples of a batch, are made ending where it ends and moved down (loadUpTo; cv_reads.h says where reads lie);
// element by element only where all vectors together are less than 16 bytes.
// Results.  A tile's results meet in the wave's own part of the LDS, whole rows or segments of them, exactly as they lie in
// memory, and leave in pieces of 16 bytes at whatever element these begin; packed vectors of any length are one block, 16 of which
// are a whole number of pieces.
// Matrix.  The whole of it lies in LDS in fragment order, one copy to a workgroup of eight waves; the row tiles are a loop, so
// that one kernel serves every number of rows (tile t: rows 16t .. 16t+15).  A matrix beyond the LDS is split by row tiles
// (blockIdx.y).
// Sums are formed as in matmulKernel and matmulLargeKernel (the same k-slots in the same instructions): the same bits.
//
// What it replaced: loads and stores of single elements wherever k, m or an address was no multiple of 16 bytes, one launch for every 128
// rows, and a matrix gathered element by element for every such launch (before, now; us): half 79 x 29 over 221 953 samples 110, 18.6;
// bfloat16 18 x 221 over 129 870 245, 22.6; int8 221 x 9 over 292 087 306, 60 (5.1 TB/s; floor 52); fp32 18 x 238 over 60 333 74, 32;
// bfloat16 156 x 211 over 16 447 144, 17.8; half 256 x 256 over 400 000 213, 119.  200 sizes between 8 and 256 over 2^10 to 2^22 samples: 2.26
// times as fast (geometric mean).  The largest are bound by HBM, small batches by launching and two trips to memory (matrix and
// vectors are requested together), those between by the trip of a tile while few waves find registers or LDS.
// Vectors staged through LDS in whole pieces took as long as read directly, 1.2 to 1.6 times for fp32 of many terms, and need the LDS.
#pragma once
#include "cv_matmul_plan.h"

namespace cv {
namespace {

// f(integral_constant<int, B>) ... f(integral_constant<int, E - 1>)
template <int B, int E, class F>
void forEach(F&& f)
{
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        forEach<B + 1, E>(f);
    }
}

__device__ __forceinline__ void meetInWave()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Lane-chunks of row tiles t0 .. t0+tb-1 to LDS, row i of tile t being row 16 t + i.  The loads of several chunks of a thread are in
// flight together: a RowMajor chunk is one read at whatever element it begins, one of a ColumnMajor matrix EPL elements.
template <class Fl, int KT, int TOGETHER, class Store>
__device__ __forceinline__ void stageRowTiles(const MatMulArgs& a, const PackedPlan& p, int t0, int tb, uint32_t gs, uint32_t xorByte, Store&& store)
{
    constexpr int EPL = Fl::kEpl, ESZ = Fl::kEsz, DW = Fl::kRawDW;
    const int chunks = tb * KT * 64, rowsLane = 4 * p.mt;
    const bool direct = fragmentSourceIsDirect<ESZ, EPL>(a.shape, a.transpose != 0, p.mt, KT, gs, (uint32_t)a.m, (uint32_t)a.k, 0, xorByte);
    const bool columns = a.shape.layout == kColumnMajor && !a.transpose;
    const size_t line = a.shape.stride ? a.shape.stride : (size_t)(columns ? a.shape.rows : a.shape.cols) * ESZ;
    for (int c0 = threadIdx.x; c0 < chunks; c0 += TOGETHER * blockDim.x) {
        uint32_t v[TOGETHER][DW];
        if (p.matBytes || columns) {
            int valid[TOGETHER];
            const uint8_t* at[TOGETHER];
#pragma unroll
            for (int u = 0; u < TOGETHER; ++u) {
                const int c = c0 + u * (int)blockDim.x, ln = c & 63, f = c >> 6;
                const uint32_t row = (uint32_t)(16 * (t0 + f / KT) + (ln & 15)), q0 = (uint32_t)(f % KT * EPL), col = (uint32_t)(ln >> 4) * gs + q0;
                valid[u] = 0;
                if (c < chunks && row < (uint32_t)a.m && q0 < gs && col < (uint32_t)a.k) valid[u] = min(min((int)(gs - q0), a.k - (int)col), EPL);
                at[u] = a.mat + (valid[u] ? columns ? (size_t)col * line + (size_t)row * ESZ : (size_t)row * line + (size_t)col * ESZ : 0);
            }
            if (columns) {
                uint32_t e[TOGETHER][EPL];
#pragma unroll
                for (int u = 0; u < TOGETHER; ++u)
#pragma unroll
                    for (int s = 0; s < EPL; ++s) {
                        const uint8_t* q = s < valid[u] ? at[u] + (size_t)s * line : a.mat;
                        if constexpr (ESZ == 4) e[u][s] = *(const uint32_t*)q;
                        else if constexpr (ESZ == 2) e[u][s] = *(const uint16_t*)q;
                        else e[u][s] = *q;
                    }
#pragma unroll
                for (int u = 0; u < TOGETHER; ++u)
#pragma unroll
                    for (int d = 0; d < DW; ++d) {
                        if constexpr (ESZ == 4) v[u][d] = e[u][d];
                        else if constexpr (ESZ == 2) v[u][d] = e[u][2 * d] | e[u][2 * d + 1] << 16;
                        else v[u][d] = e[u][4 * d] | e[u][4 * d + 1] << 8 | e[u][4 * d + 2] << 16 | e[u][4 * d + 3] << 24;
                    }
            } else {
                bool inside[TOGETHER];
#pragma unroll
                for (int u = 0; u < TOGETHER; ++u) {
                    inside[u] = (size_t)(at[u] - a.mat) + EPL * ESZ <= p.matBytes;
                    loadLoose<ESZ>(inside[u] ? at[u] : a.mat, v[u]);
                }
#pragma unroll
                for (int u = 0; u < TOGETHER; ++u)
                    if (!inside[u]) loadSlots<DW>(v[u], at[u], valid[u] * ESZ, 2);      // (the end of the last row)
            }
#pragma unroll
            for (int u = 0; u < TOGETHER; ++u) {
                if constexpr (ESZ == 1) {
#pragma unroll
                    for (int d = 0; d < DW; ++d) v[u][d] ^= xorByte * 0x01010101u;
                }
                clearBehind<ESZ>(v[u], valid[u] * ESZ);
            }
        } else {
#pragma unroll
            for (int u = 0; u < TOGETHER; ++u) {
                // (beyond the end: chunk 0 once more, which is not stored)
                const int c = c0 + u * (int)blockDim.x < chunks ? c0 + u * (int)blockDim.x : 0, ln = c & 63, f = c >> 6, kt = f % KT, row = 16 * (t0 + f / KT) + (ln & 15);
                // the place of (row, kt) in the fragment order of cv_layout.h
                const int src = (((row % rowsLane) / 4) * KT + kt) * 64 + (ln & 48) + 4 * (row / rowsLane) + (row & 3);
                fetchFragmentChunk<ESZ, EPL>(v[u], a.mat, a.shape, a.transpose != 0, direct, p.mt, KT, gs, (uint32_t)a.m, (uint32_t)a.k, 0, xorByte, src);
            }
        }
#pragma unroll
        for (int u = 0; u < TOGETHER; ++u)
            if (c0 + u * (int)blockDim.x < chunks) store(c0 + u * (int)blockDim.x, v[u]);
    }
}

// (a function that the kernel takes in: written as the kernel itself the compiler lays out its loops otherwise, 256 x 256 over 400 000 half samples 119 -> 124 us)
template <class Fl, int KT, int NT, typename OutT>
__device__ __forceinline__ void packedRows(const MatMulArgs& a, const PackedPlan& p, uint8_t* lds)
{
    constexpr int EPL = Fl::kEpl, FD = Fl::kFD, IESZ = Fl::kInEsz, IRAW = Fl::kInRawDW;
    constexpr bool F32 = kInPieces<Fl>;
    constexpr int LANE_DW = F32 ? FD : Fl::kRawDW, OESZ = sizeof(OutT);
    constexpr uint32_t S = 16 * NT;
    typedef typename Fl::Acc Acc;
    typedef typename std::conditional<Fl::kIsFloat, float, int>::type BiasT;

    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int t0 = (int)blockIdx.y * p.tb, tb = min(p.tb, p.mt - t0);
    uint32_t* const ldsW = (uint32_t*)lds;
    BiasT* const ldsBias = (BiasT*)(lds + (size_t)p.tb * KT * 64 * LANE_DW * 4);
    uint8_t* const stage = (uint8_t*)(ldsBias + 16 * p.tb) + wave * p.stageBytes;

    const uint32_t gs = optGS((uint32_t)a.k);
    const uint32_t numTiles = (uint32_t)(((uint64_t)a.batch + S - 1) / S), tileStride = gridDim.x * waves;
    uint32_t tile = blockIdx.x * waves + wave;

    // which of a lane's k-slots exist: in every lane all of the first wholeFragments fragments' ones
    const int colBase = (int)(g * gs), validBytes = sliceBytes((uint32_t)a.k, gs, g, IESZ);
    const int wholeFragments = min((int)gs, max(a.k - 3 * (int)gs, 0)) / EPL;
    constexpr bool MASK = Fl::kIsFloat || Fl::kAnySign;      // (signed bytes: what has no weight adds nothing)

    // a tile whose lanes' reads, up to the last k-slot of the last lane group, end inside the buffer
    const uint64_t inEnd = vectorsEnd(a.batch, a.inStride, (uint32_t)a.k, IESZ);
    auto inside = [&](uint32_t t) { return tileReadsEnd((uint64_t)t * S, S, a.inStride, gs, KT * EPL, IESZ) <= inEnd; };
    const int tailSlots = (int)gs - (KT - 1) * EPL, tailDwords = tailSlots * IESZ == 12 ? 4 : tailSlots * IESZ / 4;
    uint32_t raw[NT][KT][IRAW] = {};
    auto request = [&](uint32_t t) {
        const uint8_t* q = a.in + ((uint64_t)t * S + n) * a.inStride + colBase * IESZ;
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                const uint8_t* at = q + (uint64_t)(16 * j) * a.inStride + kt * EPL * IESZ;
                if (kt + 1 == KT && tailDwords < IRAW) {
                    // no more of the last fragment than some lane needs (what is not read has no weight, and is cleared)
                    if (tailDwords == 1) raw[j][kt][0] = ((const Loose4<IESZ>*)at)->v;
                    if (IRAW > 2 && tailDwords == 2) { const u32x2 v = ((const Loose8<IESZ>*)at)->v; raw[j][kt][0] = v.x; raw[j][kt][IRAW > 2 ? 1 : 0] = v.y; }
                    if (IRAW > 4 && tailDwords == 4) { const u32x4 v = ((const Loose16<IESZ>*)at)->v; raw[j][kt][0] = v.x; raw[j][kt][1] = v.y; raw[j][kt][IRAW > 4 ? 2 : 0] = v.z; raw[j][kt][IRAW > 4 ? 3 : 0] = v.w; }
                    continue;
                }
                loadLoose<IESZ>(at, raw[j][kt]);
            }
    };
    constexpr bool AHEAD = !F32 || KT <= 4;      // the next tile is requested before this one's products (registers)

    if (AHEAD && tile < numTiles && inside(tile)) request(tile);

    // ---- the block of the matrix and of the bias (whose loads overlap)
    auto biasOf = [&](int i) {
        const int row = 16 * t0 + i;
        if constexpr (Fl::kIsFloat) return (a.bias && row < a.m) ? loadAsFloat(a.bias + (size_t)row * elemSize(a.biasCt), a.biasCt) : 0.f;
        else return (a.bias && row < a.m) ? ((const int32_t*)a.bias)[row] : 0;
    };
    const BiasT firstBias = (int)threadIdx.x < 16 * tb ? biasOf(threadIdx.x) : (BiasT)0;
    bool matBeyond = false;                   // F32Mma::beyond of the matrix
    {
        uint32_t most = 0u;
        auto store = [&](int c, uint32_t (&v)[Fl::kRawDW]) {
            if constexpr (F32) {
                uint32_t pieces[FD];
                const uint32_t own = Fl::largestBits(v, 8, 0u);
                Fl::decode(v, pieces);
                if (own >= Fl::kExactBits) Fl::template decode<true>(v, pieces);
                storeFragmentChunk<FD>(ldsW + (size_t)c * FD, pieces);
                most = max(most, own);
            } else {
                storeFragmentChunk<LANE_DW>(ldsW + (size_t)c * LANE_DW, v);
            }
        };
        const uint32_t xorByte = (Fl::kAnySign && a.matUnsigned) ? 0x80u : 0u;
        if (tb * KT * 64 <= (int)blockDim.x) stageRowTiles<Fl, KT, 1>(a, p, t0, tb, gs, xorByte, store);
        else stageRowTiles<Fl, KT, Fl::kEsz == 4 ? 2 : 4>(a, p, t0, tb, gs, xorByte, store);
        if ((int)threadIdx.x < 16 * tb) ldsBias[threadIdx.x] = firstBias;
        for (int i = threadIdx.x + blockDim.x; i < 16 * tb; i += blockDim.x) ldsBias[i] = biasOf(i);
        if constexpr (F32) matBeyond = __syncthreads_or(most >= Fl::kBeyondBits);
        else __syncthreads();
        if constexpr (Fl::kAnySign) {
            if (a.inUnsigned) {               // see addUnsignedRowTerm
                for (int i = threadIdx.x; i < 16 * tb; i += blockDim.x) {
                    int sum = 0;
                    for (int f = 0; f < 4 * KT; ++f)
#pragma unroll
                        for (int d = 0; d < Fl::kRawDW; ++d) sum += sumSignedBytes(ldsW[(((i >> 4) * KT + (f >> 2)) * 64 + 16 * (f & 3) + (i & 15)) * Fl::kRawDW + d]);
                    ldsBias[i] += 128 * sum + (a.matUnsigned ? 16384 * a.k : 0);
                }
                __syncthreads();
            }
        }
    }

    while (tile < numTiles) {
        if (inside(tile)) {
            if (!AHEAD) request(tile);
        } else {
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const uint8_t* q = a.in + min((uint64_t)tile * S + 16 * j + n, (uint64_t)(a.batch - 1)) * a.inStride + colBase * IESZ;
#pragma unroll
                for (int kt = 0; kt < KT; ++kt) {
                    if (inEnd >= 16) loadUpTo<IESZ>(q + kt * EPL * IESZ, a.in + inEnd, raw[j][kt]);
                    else loadSlots<IRAW>(raw[j][kt], q + kt * EPL * IESZ, validBytes - kt * EPL * IESZ, 2);
                }
            }
        }
        int valid = validBytes;
        pinHere(valid);      // (the comparisons with it stay in the loop: hoisted, they take more scalar registers than there are)
        uint32_t b[NT][KT][FD];
        bool any[NT];
        int xSum[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            float most = 0.f;
            xSum[j] = 0;
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                uint32_t x[IRAW];
#pragma unroll
                for (int d = 0; d < IRAW; ++d) x[d] = raw[j][kt][d];
                if constexpr (Fl::kAnySign) {
#pragma unroll
                    for (int d = 0; d < IRAW; ++d) x[d] ^= a.inUnsigned ? 0x80808080u : 0u;
                }
                if (MASK && kt >= wholeFragments) clearBehind<IESZ>(x, valid - kt * EPL * IESZ);
                if constexpr (Fl::kAnySign) {
                    if (a.matUnsigned) {
#pragma unroll
                        for (int d = 0; d < IRAW; ++d) xSum[j] += sumSignedBytes(x[d]);
                    }
                }
                if constexpr (F32) most = Fl::largest(x, IRAW, most);
                Fl::decodeIn(x, b[j][kt]);
            }
            if constexpr (F32) any[j] = matBeyond | Fl::beyond(most);
            if constexpr (Fl::kAnySign) {
                if (a.matUnsigned) xSum[j] = 128 * sumOverGroups(xSum[j]);
            }
        }
        const uint32_t next = tile + tileStride;
        if (AHEAD && next < numTiles && inside(next)) request(next);

        for (int ts = 0; ts < tb; ts += p.segment) {
            const int te = min(ts + p.segment, tb);
            for (int t = ts; t < te; ++t) {
                const Acc bias = *(const Acc*)(ldsBias + 16 * t + 4 * g);
                typename SumOf<Fl>::T sum[NT];
#pragma unroll
                for (int j = 0; j < NT; ++j) sum[j] = SumOf<Fl>::start(bias);
#pragma unroll
                for (int kt = 0; kt < KT; ++kt) {
                    const uint32_t* rawW = &ldsW[((t * KT + kt) * 64 + lane) * LANE_DW];
                    uint32_t w[FD];
                    if constexpr (F32) {
#pragma unroll
                        for (int d = 0; d < FD; ++d) w[d] = rawW[d];
                    } else {
                        Fl::decode(rawW, w);
                    }
#pragma unroll
                    for (int j = 0; j < NT; ++j) sum[j] = Fl::mma(w, b[j][kt], sum[j]);
                }
                const int left = a.m - (16 * (t0 + t) + 4 * g);
                uint8_t* const o0 = stage + (uint32_t)n * p.outRow + (16 * (t - ts) + 4 * g) * OESZ;
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    Acc acc = SumOf<Fl>::finish(sum[j], bias);
                    if constexpr (F32) {
                        if (any[j]) {
                            const uint8_t* row = a.in + min((uint64_t)tile * S + 16 * j + n, (uint64_t)(a.batch - 1)) * a.inStride + (size_t)colBase * IESZ;
                            F32Careful c;
                            c.start(bias);
#pragma unroll 1
                            for (int kt = 0; kt < KT; ++kt) {
                                uint32_t x[IRAW];
                                loadSlots<IRAW>(x, row + kt * EPL * IESZ, validBytes - kt * EPL * IESZ, 1);
                                c.template step<true, false>(&ldsW[((t * KT + kt) * 64 + lane) * LANE_DW], x);
                            }
                            acc = c.finish(bias);
                        }
                    }
                    if constexpr (Fl::kAnySign) {
                        if (a.matUnsigned) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) acc[r] += xSum[j];
                        }
                    }
                    if constexpr (Fl::kIsFloat) {
                        if (a.act == kActRelu) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) acc[r] = acc[r] > 0.f ? acc[r] : 0.f;
                        } else if (a.act == kActLeakyRelu) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                if constexpr (OESZ == 2) acc[r] = activate16<OutT>(acc[r], kActLeakyRelu, a.slope);
                                else acc[r] = fmaxf(acc[r], acc[r] * a.slope);
                            }
                        } else if (a.act >= kActSigmoid) {
#pragma unroll 1
                            for (int r = 0; r < 4; ++r) {      // (one copy of their code)
                                const float x = r == 0 ? acc[0] : r == 1 ? acc[1] : r == 2 ? acc[2] : acc[3];
                                const float y = OESZ == 2 ? activate16<OutT>(x, a.act, 0.f) : smoothActivation(x, a.act);
#pragma unroll
                                for (int i = 0; i < 4; ++i) acc[i] = r == i ? y : acc[i];
                            }
                        }
                    } else {
                        if (a.act == kActRelu) {
#pragma unroll
                            for (int r = 0; r < 4; ++r) acc[r] = max(acc[r], 0);
                        }
                    }
                    uint8_t* const o = o0 + (uint32_t)(16 * j) * p.outRow;
                    if constexpr (OESZ == 2) {
                        const u32x2 v = {pack16<OutT>(acc[0], acc[1]), pack16<OutT>(acc[2], acc[3])};
                        if (left >= 4) {
                            ((Loose8<2>*)o)->v = v;
                        } else {
                            if (left > 0) ((uint16_t*)o)[0] = (uint16_t)v.x;
                            if (left > 1) ((uint16_t*)o)[1] = (uint16_t)(v.x >> 16);
                            if (left > 2) ((uint16_t*)o)[2] = (uint16_t)v.y;
                        }
                    } else {
                        const u32x4 v = __builtin_bit_cast(u32x4, acc);
                        if (left >= 4) {
                            ((Loose16<4>*)o)->v = v;
                        } else {
                            if (left > 0) ((uint32_t*)o)[0] = v.x;
                            if (left > 1) ((uint32_t*)o)[1] = v.y;
                            if (left > 2) ((uint32_t*)o)[2] = v.z;
                        }
                    }
                }
            }
            meetInWave();

            // ---- these rows' results
            const int row0 = 16 * (t0 + ts), rowsHere = min(a.m - row0, 16 * (te - ts));
            const uint32_t bytes = (uint32_t)rowsHere * OESZ;
            if (((uint64_t)tile + 1) * S <= a.batch && !p.outElements && (bytes >= 16u || !p.outPieces)) {
                uint8_t* const base = a.out + (uint64_t)tile * S * a.outStride + (size_t)row0 * OESZ;
                const uint32_t pieces = p.outPieces;
                const uint32_t last = (pieces ? S * pieces : S * bytes / 16u) - 1u;
#pragma unroll 4
                for (uint32_t c0 = 0; c0 <= last; c0 += 64) {
                    // (beyond the last piece that one again; a row's last pieces end where the row does)
                    const uint32_t c = min(c0 + lane, last), row = pieces ? (c * p.outMagic) >> 20 : 0u;
                    uint32_t at = 16u * (c - row * pieces);
                    if (pieces) at = min(at, bytes - 16u);
                    const u32x4 v = ((const Loose16<OESZ>*)(stage + row * p.outRow + at))->v;
                    uint8_t* const to = base + row * (uint32_t)a.outStride + at;
                    if (p.outLines) storeStream16(to, v);
                    else ((Loose16<OESZ>*)to)->v = v;
                }
            } else {
                // element by element: neighbouring lanes neighbouring elements of a vector
                const uint32_t first = tile * S, rows = min(S, a.batch - first);
                for (uint32_t row = 0; row < rows; ++row) {
                    OutT* dst = (OutT*)(a.out + (uint64_t)(first + row) * a.outStride) + row0;
                    for (int e = lane; e < rowsHere; e += 64) {
                        OutT v = *(const OutT*)(stage + row * p.outRow + e * OESZ);
                        if (a.accumulate) {
                            if constexpr (OESZ == 2) v = (OutT)((float)dst[e] + (float)v);
                            else v = dst[e] + v;
                        }
                        dst[e] = v;
                    }
                }
            }
            meetInWave();
        }
        tile = next;
    }
}

// waves of a workgroup: eight, of which two workgroups find the registers on a compute unit; twelve of one where fp32 operands take more
template <class Fl, int KT>
constexpr int kPackedWaves = kInPieces<Fl> && KT > 2 ? 12 : 8;
template <class Fl, int KT>
constexpr int kPackedResident = kInPieces<Fl> ? 2 : Fl::kEsz == 4 && KT > 4 ? 2 : 4;      // waves of a SIMD at least
template <class Fl, int KT, int NT, typename OutT>
__global__ __launch_bounds__((64 * kPackedWaves<Fl, KT>), (kPackedResident<Fl, KT>)) void matmulPackedKernel(const MatMulArgs a, const PackedPlan p)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    packedRows<Fl, KT, NT, OutT>(a, p, lds);
}
template <class Fl, int KT, int NT, typename OutT>
hipError_t launchPackedSized(hipStream_t stream, const MatMulArgs& a, const PackedPlan& p, uint32_t ldsBytes, int waves, int numCUs, bool append)
{
    constexpr auto kernel = matmulPackedKernel<Fl, KT, NT, OutT>;
    const hipError_t e = allowDynamicLds<kernel>((int)kPackedLds);
    if (e != hipSuccess) return e;
    int perCU = residentBlocksPerCU<kernel>(64 * kPackedWaves<Fl, KT>) * kPackedWaves<Fl, KT> / waves;
    const int byLds = (int)(kPackedLds / ldsBytes);
    if (perCU > byLds) perCU = byLds;
    const uint32_t blocksY = (uint32_t)((p.mt + p.tb - 1) / p.tb);
    const uint32_t tiles = (uint32_t)(((uint64_t)a.batch + 16 * NT - 1) / (16 * NT)), need = (tiles + waves - 1) / waves;
    uint32_t cap = (uint32_t)numCUs * (uint32_t)perCU / blocksY;
    if (cap < 1) cap = 1;
    noteKernel(append, "matmulPackedKernel<%s,KT=%d,NT=%d,out=%dB>", Fl::kName, KT, NT, (int)sizeof(OutT));
    hipLaunchKernelGGL(kernel, dim3(need < cap ? need : cap, blocksY), dim3(64 * waves), ldsBytes, stream, a, p);
    return hipGetLastError();
}

// false where the k-tiles are beyond the registers, and (whole) where the rows of a sample's results would not come from one wave at once
template <class Fl, typename OutT>
bool launchPacked(hipStream_t stream, const MatMulArgs& a, int numCUs, bool append, hipError_t& result, bool whole = false)
{
    const uint32_t kt = optKT((uint32_t)a.k, Fl::kEpl);
    constexpr int kMostKT = Fl::kEpl == 16 ? 4 : 8;
    if (kt > kMostKT) return false;
    constexpr int kMostPairs = Fl::kEsz == 4 ? 2 : 4;
    const int waves = kt > 2 ? kPackedWaves<Fl, 3> : kPackedWaves<Fl, 1>;
    const PackedCall call = {(uint32_t)a.m, kt, a.batch, (uint64_t)(uintptr_t)a.in, a.inStride, (uint64_t)a.k * Fl::kInEsz, (uint64_t)(uintptr_t)a.out, a.outStride,
                             (uint32_t)sizeof(OutT), 64u * 4u * (uint32_t)(kInPieces<Fl> ? Fl::kFD : Fl::kRawDW), kMostPairs, (uint32_t)waves, a.accumulate != 0, (uint32_t)numCUs};
    PackedLaunch l = planPacked(call);
    if (!l.fits || (whole && l.split)) return false;
    PackedPlan& p = l.plan;
    if (a.shape.layout == kRowMajor && !a.transpose) {
        p.matBytes = matrixSize(a.shape);
        if (p.matBytes < Fl::kEpl * Fl::kEsz) p.matBytes = 0;
    }
    bool done = false;
    forEach<1, kMostKT + 1>([&](auto kc) {
        constexpr int K = decltype(kc)::value;
        if ((int)kt != K) return;
        auto launch = [&](auto nc) {
            result = launchPackedSized<Fl, K, decltype(nc)::value, OutT>(stream, a, p, l.ldsBytes, waves, numCUs, append);
            done = true;
        };
        if constexpr (K <= kMostPairs) {
            if (l.nt == 2) return launch(std::integral_constant<int, 2>{});
        }
        launch(std::integral_constant<int, 1>{});
    });
    return done;
}

} // namespace
} // namespace cv
