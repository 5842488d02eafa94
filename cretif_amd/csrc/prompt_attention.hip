// prompt_attention.hip -- causal attention of a prompt's query rows over the
// [T, Hkv, D] fp32 caches (ref:src/attention.cu:809-871: Q K^T, scale, causal
// mask, softmax, P V as five launches over materialized scores), head_dim 64
// and 128, on the fp16 matrix cores at fp32 accuracy.
//
// Every fp32 operand x is scaled by a power of two into fp16's upper range and
// taken as two fp16 parts, x = hi + lo, and a product as hi hi + hi lo + lo hi,
// each exact in fp32 and summed in fp32 with the small ones first.
// v_mfma_f32_32x32x16_f16 does 16 times the multiply-adds per cycle of
// v_mfma_f32_32x32x2_f32, so the three cost 0.19 of the fp32 instruction's
// cycles.  The parts of x are off by at most 2^-23 of x or, for an x below 2^-15
// of the largest magnitude that shares its scale, 2^-38 of that magnitude (fp16's
// smallest step); lo lo, left out, is at most 2^-22 of a product and 2^-24 of it
// on average.  What operands this is enough for, and what happens to the others,
// stands with kPaSpread.  On N(0, 1) operands the outputs are 1.3 to 4 times
// closer to float64 than those of the fp32 products (launch_prompt_attention).
//
//   * prompt_kv_split_kernel writes the parts of K and V once per call, tile by
//     tile (32 positions of one KV head, D * 256 bytes), in the order the matrix
//     instructions take them: 16 bytes per lane, 64 lanes consecutive.  So a
//     tile goes to LDS with global_load_lds and comes out with conflict-free
//     16-byte reads; V is stored transposed (a lane's 8 values are 8 positions
//     of one dim).  The scale is the tile's own (its largest magnitude goes to
//     [2^13, 2^14)), one for K and one for V, kept in the tile's record.
//   * prompt_attn_kernel: a workgroup of QB x KS waves takes 32 QB queries (query
//     q = m G + g: row m, head g of the KV head's G) and the tiles they see; wave
//     (b, k) has queries 32 b .. + 31 and tiles k, k + KS, ...  The products run
//     transposed, S^T = K Q^T and O^T += V^T P^T, so a lane owns one query: its
//     16 scores of a tile are positions 8 (v >> 2) + 4 h + (v & 3), and those are
//     the positions whose probabilities it supplies to O^T, so P never leaves the
//     registers.  The scores of the wave's next tile are issued between the
//     softmax instructions of the current one; the tiles of the stage after are
//     copied meanwhile (K and V double-buffered, one barrier per stage).
//   * probabilities enter O^T times 2^kShift (and a factor that evens out the V
//     scales: all accumulators are in units of the largest V tile the workgroup
//     sees).  The running maximum is only raised, and the accumulators rescaled,
//     when a score exceeds it by more than kSlack, so after the first tiles the
//     rescale is rarely taken; 2^(kShift + kSlack) is inside fp16.
//   * the KS waves of a query block meet in LDS in wave order and the workgroup
//     writes the output, or, where few query groups leave the GPU idle and the
//     positions are cut into chunks, one (max, sum, acc) record per (row, head,
//     chunk) for the combine kernel of the decode attention.
//
// A workgroup whose queries or tiles are not of that kind (kPaSpread), or lie near
// the ends of fp32's range (a tile of K or V, or a query, holding an infinity, a
// NaN or a value of 2^60, or whose largest magnitude is below 2^-50), takes fp32
// products from the caches on v_mfma_f32_32x32x2_f32 instead (plain_group).
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "common.hpp"
#include "internal.hpp"

namespace cri {
namespace dev {
namespace {

typedef _Float16 pah2 __attribute__((ext_vector_type(2)));
typedef _Float16 pah8 __attribute__((ext_vector_type(8)));
typedef float paf2 __attribute__((ext_vector_type(2)));
typedef float paf16 __attribute__((ext_vector_type(16)));

constexpr int kPaTile = 32;       // positions per tile
constexpr int kShift = 12;        // log2 of the probabilities' scale
constexpr float kSlack = 3.0f;    // base-2 headroom of a score over the running maximum
// bits of 2^60 and 2^-50: scale exponents from -46 to 63, so that the product of two scales, of a tile
// that is seen or not, and 2^(kShift - a difference of two) are normal numbers (a score's factor of 0 or
// infinity would meet masked scores of -infinity and scores of 0)
constexpr uint32_t kPaMax = 0x5D800000u, kPaMin = 0x26800000u;
// The parts' fixed steps must not show beside fp32's rounding (2^-24):
//   * a score is off by at most D 2^-37 of (largest |q|) (largest |k|), an amount that a score of
//     fewer or smaller terms may notice; in base 2, where it counts as it is, that is 2^-21 at worst
//     (aligned signs; 2^-26 as a root of D) while the product is below 2^kPaScore;
//   * a probability is off by 2^-37 of the largest, so values may be at most 2^kPaSpread apart between the
//     rows (and dims) a workgroup meets: then the large ones' share is off by 2^-27 of the small ones;
//   * a value is off by 2^-38 of its tile's largest: 2^-28 of its own row's and dim's largest (a single value
//     far below both is less exact than in fp32, by an amount that does not show in its row).
// Measured with dims of K or V 2^8 apart, rows of V 2^8 apart, rows of K 2^6 apart or queries' dims 2^6 apart: 0.2 to
// 0.8 of the fp32 products' error, in the 2-norm and in the largest error over the sum of an output's terms.
// Rows and dims of zeros do not count, and dims only in tiles of at least kPaDimRows rows (with fewer, a
// dim's largest is small by chance).
constexpr int kPaSpread = 10;
constexpr int kPaScore = 10;
constexpr int kPaDimRows = 4;
constexpr int kPaNoScale = 1 << 20;  // a tile of zeros
constexpr int kPaZeroExp = 63;       // scale exponent of zeros: as of the smallest magnitudes
constexpr int kPaXcds = 8;

__host__ __device__ constexpr long pa_tile_bytes(int D) { return static_cast<long>(D) * 256; }

// a tile's record
struct PaTile {
    float kf;  // 2^-(K scale exponent)
    int ve;    // V scale exponent, kPaNoScale for zeros
    int vs;    // the scale exponent of V's row or dim of the smallest largest magnitude
    int bad;
};

// the two fp16 parts of the pair (a f, b f), f a power of two, each packed in a dword (the lo
// parts are one v_fma_mix each)
__device__ __forceinline__ void split2(float a, float b, float f, uint32_t& hi, uint32_t& lo) {
    const paf2 x = {a * f, b * f};
    const pah2 p = __builtin_convertvector(x, pah2);
    const pah2 r = {static_cast<_Float16>(__builtin_fmaf(a, f, -static_cast<float>(p.x))),
                    static_cast<_Float16>(__builtin_fmaf(b, f, -static_cast<float>(p.y)))};
    hi = __builtin_bit_cast(uint32_t, p);
    lo = __builtin_bit_cast(uint32_t, r);
}

__device__ __forceinline__ void split2x8(const float (&x)[8], float f, u32x4 (&p)[2]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        uint32_t a, b;
        split2(x[2 * e], x[2 * e + 1], f, a, b);
        p[0][e] = a;
        p[1][e] = b;
    }
}

__device__ __forceinline__ paf16 mma(const u32x4& a, const u32x4& b, const paf16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(pah8, a), __builtin_bit_cast(pah8, b), c, 0, 0, 0);
}

// magnitudes are compared as bit patterns, which order as the floats do with NaN above infinity
__device__ __forceinline__ uint32_t absbits(float x) { return __builtin_bit_cast(uint32_t, x) & 0x7FFFFFFFu; }
// Reductions on the VALU alone (a __shfl_xor is a trip through the LDS pipe): quad permutations, rotations of
// 16-lane rows, and exchanges of rows and half-waves.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_bits(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), CTRL, 0xF, 0xF, false));
}
constexpr int kRowRor4 = 0x124, kRowRor8 = 0x128;
__device__ __forceinline__ uint32_t max32(uint32_t v) {  // with lane ^ 32
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return max(static_cast<uint32_t>(r[0]), static_cast<uint32_t>(r[1]));
}
// even 16-lane rows: the larger of a and lane + 16's a; odd ones: of b and lane - 16's b
__device__ __forceinline__ uint32_t max16(uint32_t a, uint32_t b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    return max(static_cast<uint32_t>(r[0]), static_cast<uint32_t>(r[1]));
}
__device__ __forceinline__ uint32_t wave_max_bits(uint32_t v) {
    v = max(v, dpp_bits<kQuadPerm1032>(v));
    v = max(v, dpp_bits<kQuadPerm2301>(v));
    v = max(v, dpp_bits<kRowRor4>(v));
    v = max(v, dpp_bits<kRowRor8>(v));
    return max32(max16(v, v));
}
// the larger of the lanes' a (bit m of the lane clear) or b (set), CTRL exchanging lanes that differ in m alone
template <int CTRL>
__device__ __forceinline__ uint32_t halve_max(uint32_t a, uint32_t b, bool set) {
    return max(set ? b : a, dpp_bits<CTRL>(set ? a : b));
}
__device__ __forceinline__ int wave_max_int(int v) {
    return static_cast<int>(wave_max_bits(static_cast<uint32_t>(v) ^ 0x80000000u) ^ 0x80000000u);
}
// true when the parts of values with this largest magnitude are not good to 2^-24
__device__ __forceinline__ bool out_of_range(uint32_t m) { return m >= kPaMax || (m != 0 && m < kPaMin); }
// exponent that brings a largest magnitude m (in range) to [2^13, 2^14)
__device__ __forceinline__ int scale_exp(uint32_t m) { return m ? 13 + 127 - static_cast<int>(m >> 23) : kPaZeroExp; }
__device__ __forceinline__ float pow2(int e) { return __builtin_bit_cast(float, (e + 127) << 23); }  // |e| <= 126

// 16 bytes per lane from global memory into LDS (lane l at byte 16 l of the wave-uniform lds)
__device__ __forceinline__ void pa_dma16(const char* g, char* lds) { __builtin_amdgcn_global_load_lds(g, lds, 16, 0, 0); }

// One tile of one KV head: K parts at byte (part * D / 16 + ks) * 1024 + 16 lane (lane (i, h):
// key i, dims 16 ks + 8 h .. + 7), V parts at D * 128 + ((part * D / 32 + db) * 2 + s) * 1024 +
// 16 lane (lane (i, h): dim 32 db + i, positions 16 s + 8 (e >> 2) + 4 h + (e & 3), e = 0 .. 7).
// Positions from T on are zeros.  Bound by memory: 8 bytes read and 8 written per position and dim.
template <int D>
__global__ __launch_bounds__(4 * D) void prompt_kv_split_kernel(const float* __restrict__ Kc,
                                                                const float* __restrict__ Vc, char* __restrict__ tiles,
                                                                PaTile* __restrict__ recs, int n_kv, int ntiles,
                                                                const int* __restrict__ kv_dev, int kv0, int M) {
    constexpr int kW = 4 * D / 64;
    __shared__ uint32_t red[2][kW];
    __shared__ uint32_t rows[D / 32][32], cols[2][D];  // largest magnitudes of V's rows and dims, in parts
    const int T = (kv_dev ? *kv_dev : 0) + kv0 + M - 1;
    const int tile = blockIdx.x, kv = blockIdx.y, t0 = tile * kPaTile;
    if (t0 >= T) return;
    char* const out = tiles + (static_cast<long>(kv) * ntiles + tile) * pa_tile_bytes(D);
    const long row = static_cast<long>(n_kv) * D;
    const int t = threadIdx.x, lane = t & 63, f = t >> 6;
    const int c = t % (D / 8), i = t / (D / 8);  // K: dims 8 c .. + 7 of key i
    float k[8], v[8];
    uint32_t km = 0, vm = 0;
    const float* src = Kc + static_cast<long>(min(t0 + i, T - 1)) * row + kv * D + 8 * c;
    const f32x4 a = ld_f32x4(src), b = ld_f32x4(src + 4);
#pragma unroll
    for (int e = 0; e < 8; ++e) {  // V: dim 32 (f / 2) + lane & 31, the positions of fragment f & 1
        const int pos = t0 + 16 * (f & 1) + 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
        v[e] = Vc[static_cast<long>(min(pos, T - 1)) * row + kv * D + 32 * (f >> 1) + (lane & 31)];
        if (pos >= T) v[e] = 0.0f;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        k[e] = t0 + i < T ? a[e] : 0.0f;
        k[4 + e] = t0 + i < T ? b[e] : 0.0f;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        km = max(km, absbits(k[e]));
        vm = max(vm, absbits(v[e]));
    }
    {
        // a row of V: over the wave's 32 dims; the lanes end with the value e of their bits 4, 0 and 1
        uint32_t x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = max16(absbits(v[e]), absbits(v[4 + e]));
        x[0] = halve_max<kQuadPerm1032>(x[0], x[2], lane & 1);
        x[1] = halve_max<kQuadPerm1032>(x[1], x[3], lane & 1);
        x[0] = halve_max<kQuadPerm2301>(x[0], x[1], lane & 2);
        x[0] = max(x[0], dpp_bits<kRowRor8>(x[0]));
        x[0] = max(x[0], dpp_bits<kRowRor4>(x[0]));
        if ((lane & 12) == 0)  // e = 4 (bit 4) + 2 (bit 0) + (bit 1)
            rows[f >> 1][16 * (f & 1) + 8 * ((lane >> 4) & 1) + 4 * (lane >> 5) + 2 * (lane & 1) +
                         ((lane >> 1) & 1)] = x[0];
    }
    vm = max32(vm);
    if (lane < 32) cols[f & 1][32 * (f >> 1) + lane] = vm;
    km = wave_max_bits(km);
    vm = wave_max_bits(vm);
    if (lane == 0) {
        red[0][f] = km;
        red[1][f] = vm;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kW; ++w) {
        km = max(km, red[0][w]);
        vm = max(vm, red[1][w]);
    }
    const bool bad = out_of_range(km) || out_of_range(vm);
    const int ke = bad ? 0 : scale_exp(km), ve = bad ? 0 : scale_exp(vm);
    u32x4 p[2];
    if (bad) {  // zeros: a wave may multiply the probabilities 0 of a tile none of its queries sees
#pragma unroll
        for (int e = 0; e < 8; ++e) k[e] = v[e] = 0.0f;
    }
    split2x8(k, pow2(ke), p);
#pragma unroll
    for (int q = 0; q < 2; ++q)
        *reinterpret_cast<u32x4*>(out + (q * (D / 16) + (c >> 1)) * 1024 + 16 * (32 * (c & 1) + i)) = p[q];
    split2x8(v, pow2(ve), p);
#pragma unroll
    for (int q = 0; q < 2; ++q)
        *reinterpret_cast<u32x4*>(out + D * 128 + (q * (D / 16) + f) * 1024 + 16 * lane) = p[q];
    if (f == 0) {
        uint32_t inv = 0;  // ~(the least of the largest magnitudes of V's rows and dims but those of zeros)
        auto take = [&](uint32_t x) { inv = max(inv, x ? ~x : 0u); };
        if (T - t0 >= kPaDimRows) {
#pragma unroll
            for (int d = lane; d < D; d += 64) take(max(cols[0][d], cols[1][d]));
        }
        uint32_t r0 = 0;
#pragma unroll
        for (int x = 0; x < D / 32; ++x) r0 = max(r0, rows[x][lane & 31]);
        take(r0);
        inv = wave_max_bits(inv);
        if (t == 0) {
            PaTile r;
            r.kf = pow2(-ke);
            r.ve = vm ? ve : kPaNoScale;
            r.vs = scale_exp(~inv);
            r.bad = bad;
            recs[kv * ntiles + tile] = r;
        }
    }
}

struct PromptArgs {
    const float* Q;
    const float* K;
    const float* V;
    const char* tiles;
    const PaTile* recs;
    const int* kv_dev;
    float* out;  // direct output (nchunks == 1), rows ldo floats apart
    float* part;  // chunk records otherwise
    long ldq, ldo;
    int kv0, M, G, n_kv, ntiles, nchunks, paired;
    float qscale;  // scale * log2 e: scores are in base 2
};

// floats of one query's record in the merge area (row stride that spreads the banks)
constexpr int pa_row(int D) { return D + 4; }

template <int D, int QB, int KS>
constexpr int pa_lds_bytes() {
    constexpr int stage = 2 * KS * static_cast<int>(pa_tile_bytes(D));  // K and V of KS tiles, twice
    constexpr int merge = (KS - 1) * QB * 32 * (pa_row(D) * 4 + 8);
    return stage > merge ? stage : merge;
}

template <int D, int QB, int KS>
__global__ __launch_bounds__(64 * QB * KS) __attribute__((amdgpu_waves_per_eu(2, 2))) void prompt_attn_kernel(
    const PromptArgs a) {
    constexpr int kWaves = QB * KS, kKs = D / 16, kDb = D / 32, kHalf = D * 128;  // bytes of a tile's K or V
    constexpr int kCopies = kHalf / 1024, kBuf = KS * kHalf;
    extern __shared__ __attribute__((aligned(16))) char lds[];  // K twice, V twice, KS tiles each
    const int tid = threadIdx.x, lane = tid & 63, i = lane & 31, h = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), b = w / KS, kw = w % KS;
    const int nq = a.M * a.G, ngrp = (nq + 32 * QB - 1) / (32 * QB);
    const int nb = static_cast<int>(gridDim.x), bid = static_cast<int>(blockIdx.x);
    // each XCD (workgroup id mod 8) takes a contiguous range of the work, so a KV head's tiles are
    // read through one L2
    const int wi = nb % kPaXcds == 0 ? (bid % kPaXcds) * (nb / kPaXcds) + bid / kPaXcds : bid;
    // paired (one chunk): a workgroup takes a KV head's p-th longest query group, then its p-th
    // shortest, so every workgroup does about the same work
    const int per_kv = a.paired ? (ngrp + 1) / 2 : ngrp * a.nchunks;
    const int kvh = wi / per_kv, r0 = wi % per_kv;
    const int c = a.paired ? 0 : r0 / ngrp;
    const int grp0 = ngrp - 1 - (a.paired ? r0 : r0 % ngrp);
    const int Tb = (a.kv_dev ? *a.kv_dev : 0) + a.kv0;  // row m attends to positions [0, Tb + m)
    const int Tmax = Tb + a.M - 1;
    constexpr int kStagePos = kPaTile * KS;
    const int Tc = kStagePos * (((Tmax + kStagePos - 1) / kStagePos + a.nchunks - 1) / a.nchunks);
    const int t0 = c * Tc, t1 = min(Tmax, t0 + Tc);
    const char* const tiles = a.tiles + static_cast<long>(kvh) * a.ntiles * pa_tile_bytes(D);
    // the tile records, read with scalar loads
    typedef const __attribute__((address_space(4))) PaTile* RecPtr;
    const RecPtr recs = (RecPtr)(a.recs + static_cast<long>(kvh) * a.ntiles);
    const int first_tile = t0 / kPaTile, last_tile = (Tmax - 1) / kPaTile;

    // the waves of a query block meet in wave order: waves kw > 0 through LDS into wave 0, which writes the sums of
    // the lanes' queries (row qm, head qg; o times back)
    auto merge = [&](const float mx, const float l, paf16 (&o)[kDb], int qm, int qg, bool qok, float back) {
        const float lq = l + shfl_xor32(l);
        float* const mg = reinterpret_cast<float*>(lds);
        float* const ml = mg + (KS - 1) * QB * 32 * pa_row(D);
        __syncthreads();
        if (kw > 0) {
            const int slot = ((kw - 1) * QB + b) * 32 + i;
            float* dst = mg + slot * pa_row(D) + 4 * h;
#pragma unroll
            for (int d = 0; d < kDb; ++d)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    *reinterpret_cast<f32x4*>(dst + 32 * d + 8 * v) =
                        f32x4{o[d][4 * v], o[d][4 * v + 1], o[d][4 * v + 2], o[d][4 * v + 3]};
            if (h == 0) {
                ml[2 * slot] = mx;
                ml[2 * slot + 1] = lq;
            }
        }
        __syncthreads();
        if (kw == 0 && qok) {
            float M = mx;
#pragma unroll
            for (int x = 0; x < KS - 1; ++x) M = fmaxf(M, ml[2 * ((x * QB + b) * 32 + i)]);
            float f = mx == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mx - M);
            float L = f * lq;
#pragma unroll
            for (int d = 0; d < kDb; ++d) o[d] *= f;
#pragma unroll
            for (int x = 0; x < KS - 1; ++x) {
                const int slot = (x * QB + b) * 32 + i;
                const float mo = ml[2 * slot];
                f = mo == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mo - M);
                L = __builtin_fmaf(f, ml[2 * slot + 1], L);
                const float* src = mg + slot * pa_row(D) + 4 * h;
#pragma unroll
                for (int d = 0; d < kDb; ++d)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const f32x4 y = *reinterpret_cast<const f32x4*>(src + 32 * d + 8 * v);
#pragma unroll
                        for (int e = 0; e < 4; ++e) o[d][4 * v + e] = __builtin_fmaf(f, y[e], o[d][4 * v + e]);
                    }
            }
            const int head = kvh * a.G + qg;
            float* dst;
            if (a.out) {
                dst = a.out + qm * a.ldo + static_cast<long>(head) * D + 4 * h;
            } else {
                float* r = a.part + ((static_cast<long>(qm) * a.G * a.n_kv + head) * a.nchunks + c) * (D + 4);
                if (h == 0) {
                    r[0] = M;
                    r[1] = L;
                }
                dst = r + 4 + 4 * h;
            }
            const float den = a.out ? L : 1.0f;
#pragma unroll
            for (int d = 0; d < kDb; ++d)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    f32x4 y;
#pragma unroll
                    for (int e = 0; e < 4; ++e) y[e] = o[d][4 * v + e] / den * back;
                    *reinterpret_cast<f32x4*>(dst + 32 * d + 8 * v) = y;
                }
        }
    };

    // one query group; false (and nothing written) where its operands are not for the parts
    auto run_group = [&](const int grp) {
        const int q0 = grp * 32 * QB + 32 * b;  // the wave's queries q0 .. q0 + 31
        const int q = q0 + i;
        const bool qok = q < nq;
        const int qm = qok ? q / a.G : 0, qg = qok ? q - qm * a.G : 0;
        const int lim = qok ? min(Tb + qm, t1) : t1;  // positions below lim are visible
        // the wave's first limit and the workgroup's last
        const int lim_lo = min(Tb + min(q0, nq - 1) / a.G, t1);
        const int end = min(Tb + min(grp * 32 * QB + 32 * QB - 1, nq - 1) / a.G, t1);
        const int nst = end > t0 ? (end - t0 + kStagePos - 1) / kStagePos : 0;

        u32x4 qf[2][kKs];  // B operand of S^T: the query's dims 16 ks + 8 h .. + 7, scaled into base 2
        float qinv;        // 2^-(the query's scale exponent)
        uint32_t qmx = 0;
        {
            const float* qp = a.Q + qm * a.ldq + static_cast<long>(kvh * a.G + qg) * D + 8 * h;
            float x[kKs][8];
#pragma unroll
            for (int ks = 0; ks < kKs; ++ks) {
                const f32x4 u = ld_f32x4(qp + 16 * ks) * a.qscale, v = ld_f32x4(qp + 16 * ks + 4) * a.qscale;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x[ks][e] = qok ? u[e] : 0.0f;
                    x[ks][4 + e] = qok ? v[e] : 0.0f;
                }
            }
#pragma unroll
            for (int ks = 0; ks < kKs; ++ks)
#pragma unroll
                for (int e = 0; e < 8; ++e) qmx = max(qmx, absbits(x[ks][e]));
            qmx = max32(qmx);
            const int qe = out_of_range(qmx) ? 0 : scale_exp(qmx);
            qinv = pow2(-qe);
#pragma unroll
            for (int ks = 0; ks < kKs; ++ks) {
                u32x4 p[2];
                split2x8(x[ks], pow2(qe), p);
                qf[0][ks] = p[0];
                qf[1][ks] = p[1];
            }
        }
        // the records of every tile the workgroup sees: a flag, or magnitudes too far apart, or scores too
        // large, or queries out of range take the fp32 path; E is the scale of the accumulators
        int E;
        {
            bool slow = out_of_range(qmx);
            uint32_t kfm = 0;  // bits of the factor of the largest |k|
            int lo = -(1 << 20), hi = -(1 << 20);  // -(least exponent), largest exponent
            const PaTile* r = a.recs + static_cast<long>(kvh) * a.ntiles;
            for (int t = first_tile + lane; t * kPaTile < end; t += 64) {
                slow |= r[t].bad != 0;
                kfm = max(kfm, absbits(r[t].kf));
                if (r[t].ve != kPaNoScale) {
                    lo = max(lo, -r[t].ve);
                    hi = max(hi, r[t].vs);
                }
            }
            kfm = wave_max_bits(kfm);
            // the magnitudes are below 2^14 times qinv and kfm
            slow |= qinv * __builtin_bit_cast(float, kfm) > pow2(kPaScore - 28);
            lo = -wave_max_int(lo);
            hi = wave_max_int(hi);
            E = __builtin_amdgcn_readfirstlane(lo == 1 << 20 ? 0 : lo);
            slow |= hi - lo > kPaSpread;
            if (__syncthreads_or(slow)) return false;  // (also: the previous group's merge has been read)
        }

        // the K or V half of stage st's tiles into buffer st & 1; the waves share the copies
        auto copy = [&](int st, bool v) {
            char* const buf = lds + (v ? 2 * kBuf : 0) + (st & 1) * kBuf;
#pragma unroll
            for (int n = 0; n < KS * kCopies / kWaves; ++n) {
                const int x = n * kWaves + w, t = x / kCopies, o = (x % kCopies) * 1024;
                const int tile = min(first_tile + st * KS + t, last_tile);
                pa_dma16(tiles + tile * pa_tile_bytes(D) + (v ? kHalf : 0) + o + 16 * lane, buf + t * kHalf + o);
            }
        };
        static_assert(KS * kCopies % kWaves == 0, "the waves share a stage's copies evenly");
        auto rec_of = [&](int st) { return min(first_tile + st * KS + kw, last_tile); };
        float mx = -INFINITY, l = 0.0f;
        paf16 o[kDb];
#pragma unroll
        for (int d = 0; d < kDb; ++d)
#pragma unroll
            for (int v = 0; v < 16; ++v) o[d][v] = 0.0f;
        // scores s (times 1 / f) of the tile at tb: mask, and the running maximum
        auto raise = [&](int tb, float f, paf16& s) {
            if (tb + kPaTile > lim_lo) {
                const int rel = lim - tb - 4 * h;
#pragma unroll
                for (int v = 0; v < 16; ++v) s[v] = 8 * (v >> 2) + (v & 3) < rel ? s[v] : -INFINITY;
            }
            float tmax = s[0];
#pragma unroll
            for (int v = 1; v < 16; ++v) tmax = fmaxf(tmax, s[v]);
            tmax = fmaxf(tmax, shfl_xor32(tmax)) * f;  // with the query's other 16 positions
            if (__any(tmax > mx + kSlack)) {           // (mx = -inf: any visible position)
                const float mnew = fmaxf(mx, tmax);
                const float cf = mnew == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mx - mnew);
                mx = mnew;
                l *= cf;
#pragma unroll
                for (int d = 0; d < kDb; ++d) o[d] *= cf;
            }
        };
        // One block of MFMAs and VALU, one MFMA per few VALU instructions: the next tile's scores
        // sn = S^T from kt (hi lo and lo hi first: the larger sums are rounded last) and, from the scores
        // s, the probabilities 2^(s f - base), times pscale as the B operand of O^T (parts of position
        // block 16 k: pf[part][k]).  (first: only the scores, of the first tile)
        u32x4 pf[2][2];
        auto block = [&](const char* kt, const paf16& s, float f, float base, float pscale, paf16& sn,
                         auto first) {
#pragma unroll
            for (int v = 0; v < 16; ++v) sn[v] = 0.0f;
#pragma unroll
            for (int ks = 0; ks < kKs; ++ks) {
                const u32x4 k0 = *reinterpret_cast<const u32x4*>(kt + ks * 1024);
                const u32x4 k1 = *reinterpret_cast<const u32x4*>(kt + (kKs + ks) * 1024);
                sn = mma(k1, qf[0][ks], sn);
                sn = mma(k0, qf[1][ks], sn);
                if constexpr (!decltype(first)::value) {
                    constexpr int kPer = 16 / kKs;  // scores per 16 dims
                    float x[kPer];
#pragma unroll
                    for (int e = 0; e < kPer; ++e) {
                        x[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kPer * ks + e], f, -base));
                        l += x[e];
                    }
#pragma unroll
                    for (int e = 0; e < kPer; e += 2) {
                        const int v = kPer * ks + e;
                        uint32_t p0, p1;
                        split2(x[e], x[e + 1], pscale, p0, p1);
                        pf[0][v >> 3][(v & 7) >> 1] = p0;
                        pf[1][v >> 3][(v & 7) >> 1] = p1;
                    }
                }
            }
            // head_dim 128: the hi parts of K are read again instead of being kept (32 registers)
            if constexpr (kKs > 4) asm volatile("" ::: "memory");
#pragma unroll
            for (int ks = 0; ks < kKs; ++ks) sn = mma(*reinterpret_cast<const u32x4*>(kt + ks * 1024), qf[0][ks], sn);
            if constexpr (!decltype(first)::value) {
#pragma unroll
                for (int n = 0; n < 3 * kKs; ++n) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                // MFMA
                    __builtin_amdgcn_sched_group_barrier(0x402, kKs == 4 ? 8 : 4, 0);  // VALU
                }
            }
        };
        auto values = [&](const char* vt) {
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int d = 0; d < kDb; ++d) {
                    const u32x4 v0 = *reinterpret_cast<const u32x4*>(vt + (d * 2 + k) * 1024);
                    const u32x4 v1 = *reinterpret_cast<const u32x4*>(vt + ((kDb + d) * 2 + k) * 1024);
                    o[d] = mma(v1, pf[0][k], o[d]);
                    o[d] = mma(v0, pf[1][k], o[d]);
                    o[d] = mma(v0, pf[0][k], o[d]);
                }
        };
        // every wave waits for its own copies before a barrier; the barrier also orders the reads of a
        // buffer before the next copy into it
        auto arrive = [&]() {
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
            __syncthreads();
        };
        const char* const mine = lds + kw * kHalf + 16 * lane;
        int tb = t0 + kw * kPaTile;
        // stage st (position J = st & 1 of the buffers); r: its tile's record, the next one's when it returns
        auto stage = [&](int st, auto pos, float& kf, int& ve, paf16& s, paf16& sn) {
            constexpr int J = decltype(pos)::value;
            const RecPtr rn = recs + rec_of(st + 1);
            const float kfn = rn->kf;
            const int ven = rn->ve;
            arrive();  // K of stage st + 1 and V of stage st; every read of stage st - 1 is done
            if (st + 2 < nst) copy(st + 2, false);
            if (st + 1 < nst) copy(st + 1, true);
            const float f = qinv * kf;
            raise(tb, f, s);
            const int de = ve == kPaNoScale ? 0 : ve - E;  // 0 .. kPaSpread
            const float base = mx == -INFINITY ? 0.0f : mx;
            block(mine + (1 - J) * kBuf, s, f, base, pow2(kShift - de), sn, std::false_type{});
            values(mine + 2 * kBuf + J * kBuf);
            kf = kfn;
            ve = ven;
            tb += kStagePos;
        };
        if (nst > 0) {
            paf16 s0, s1;
            float kf = recs[rec_of(0)].kf;
            int ve = recs[rec_of(0)].ve;
            copy(0, false);
            copy(0, true);
            if (nst > 1) copy(1, false);
            arrive();
            block(mine, s1, 0.0f, 0.0f, 0.0f, s0, std::true_type{});
            for (int st = 0;; st += 2) {
                stage(st, std::integral_constant<int, 0>{}, kf, ve, s0, s1);
                if (st + 1 >= nst) break;
                stage(st + 1, std::integral_constant<int, 1>{}, kf, ve, s1, s0);
                if (st + 2 >= nst) break;
            }
        }

        merge(mx, l, o, qm, qg, qok, pow2(-E - kShift));
        return true;
    };
    // The same group with fp32 products, in the same transposed layout: the n-th instruction of S^T takes dim
    // 8 (n >> 2) + 4 h + (n & 3) from lane (i, h) for key i and query i, the n-th of a dim block of O^T position
    // 8 (n >> 2) + 4 h + (n & 3), whose probability the lane holds in its n-th score.  Bound by the matrix
    // instructions and, its loads hidden by the SIMD's other wave only, their latency: every query of 2048 rows,
    // 32/8 heads of 64, 250 us (the five launches over materialized scores 591, one query at a time on scalar
    // FMAs 18300); heads of 128 490 (768, 33500); 64 rows 17 (32, 262).
    auto plain_group = [&](const int grp) {
        const int q0 = grp * 32 * QB + 32 * b, q = q0 + i;
        const bool qok = q < nq;
        const int qm = qok ? q / a.G : 0, qg = qok ? q - qm * a.G : 0;
        const int lim = qok ? min(Tb + qm, t1) : t1, lim_lo = min(Tb + min(q0, nq - 1) / a.G, t1);
        float mx = -INFINITY, l = 0.0f;
        paf16 o[kDb];
#pragma unroll
        for (int d = 0; d < kDb; ++d)
#pragma unroll
            for (int v = 0; v < 16; ++v) o[d][v] = 0.0f;
        const long row = static_cast<long>(a.n_kv) * D;
        const float *const Kh = a.K + kvh * D + 4 * h, *const Vh = a.V + kvh * D;
        const float* const qp = a.Q + qm * a.ldq + static_cast<long>(kvh * a.G + qg) * D + 4 * h;
        float* const ps = reinterpret_cast<float*>(lds) + w * 2048;  // [32 positions][32 queries], then [..][dims]
        static_assert(pa_lds_bytes<D, QB, KS>() >= kWaves * 8192);
        const int hi = q0 < nq ? min(Tb + min(q0 + 31, nq - 1) / a.G, t1) : t0;  // the wave's last limit
        for (int tb = t0 + kw * kPaTile; tb < hi; tb += kStagePos) {
            const float* const kp = Kh + min(tb + i, Tmax - 1) * row;
            paf16 sa, sb;  // two chains
#pragma unroll
            for (int v = 0; v < 16; ++v) sa[v] = sb[v] = 0.0f;
#pragma unroll
            for (int c = 0; c < D / 64; ++c) {
                // (the query is read again for every tile: at head_dim 128 there is no room to keep it)
                if constexpr (D > 64) asm volatile("" ::: "memory");
                f32x4 k[8], qv[8];
#pragma unroll
                for (int n = 0; n < 8; ++n) k[n] = ld_f32x4(kp + 64 * c + 8 * n);
#pragma unroll
                for (int n = 0; n < 8; ++n) qv[n] = ld_f32x4(qp + 64 * c + 8 * n);
#pragma unroll
                for (int n = 0; n < 8; ++n) {
                    sa = __builtin_amdgcn_mfma_f32_32x32x2f32(k[n].x, qv[n].x, sa, 0, 0, 0);
                    sb = __builtin_amdgcn_mfma_f32_32x32x2f32(k[n].y, qv[n].y, sb, 0, 0, 0);
                    sa = __builtin_amdgcn_mfma_f32_32x32x2f32(k[n].z, qv[n].z, sa, 0, 0, 0);
                    sb = __builtin_amdgcn_mfma_f32_32x32x2f32(k[n].w, qv[n].w, sb, 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            float p[16], tmax = -INFINITY;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                p[v] = tb + 8 * (v >> 2) + 4 * h + (v & 3) < lim ? (sa[v] + sb[v]) * a.qscale : -INFINITY;
                tmax = fmaxf(tmax, p[v]);
            }
            const float mnew = fmaxf(mx, fmaxf(tmax, shfl_xor32(tmax)));
            const float base = mnew == -INFINITY ? 0.0f : mnew;
            const float cf = __builtin_amdgcn_exp2f(mx - base);
            mx = mnew;
            l *= cf;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                p[v] = __builtin_amdgcn_exp2f(p[v] - base);
                l += p[v];
            }
#pragma unroll
            for (int d = 0; d < kDb; ++d) o[d] *= cf;
#pragma unroll
            for (int d0 = 0; d0 < kDb; d0 += 2) {
                float x[2][16];
                bool odd = false;
#pragma unroll
                for (int n = 0; n < 16; ++n) {
                    const float* const vp =
                        Vh + min(tb + 8 * (n >> 2) + 4 * h + (n & 3), Tmax - 1) * row + 32 * d0 + i;
#pragma unroll
                    for (int d = 0; d < 2; ++d) {
                        x[d][n] = vp[32 * d];
                        odd |= absbits(x[d][n]) >= 0x7F800000u;
                    }
                }
                if (tb + kPaTile > lim_lo && __any(odd)) {
                    // an infinite or NaN value that not every query sees: times the probability 0 of those
                    // that do not, it would reach them
#pragma unroll
                    for (int d = 0; d < 2; ++d) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            ps[32 * (8 * (v >> 2) + 4 * h + (v & 3)) + i] = p[v];
                            ps[32 * (32 + 8 * (v >> 2) + 4 * h + (v & 3)) + i] = x[d][v];
                        }
                        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                        __builtin_amdgcn_wave_barrier();
#pragma unroll 4
                        for (int u = 0; u < kPaTile; ++u) {
                            const float pu = ps[32 * u + i];
                            const uint32_t seen = tb + u < lim ? ~0u : 0u;  // (a select would become branches)
#pragma unroll
                            for (int v = 0; v < 4; ++v) {
                                const u32x4 y =
                                    *reinterpret_cast<const u32x4*>(ps + 32 * (32 + u) + 8 * v + 4 * h) & seen;
                                const f32x4 z = __builtin_bit_cast(f32x4, y);
#pragma unroll
                                for (int e = 0; e < 4; ++e)
                                    o[d0 + d][4 * v + e] = __builtin_fmaf(pu, z[e], o[d0 + d][4 * v + e]);
                            }
                        }
                        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                        __builtin_amdgcn_wave_barrier();
                    }
                } else {
#pragma unroll
                    for (int n = 0; n < 16; ++n)
#pragma unroll
                        for (int d = 0; d < 2; ++d)
                            o[d0 + d] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[d][n], p[n], o[d0 + d], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        merge(mx, l, o, qm, qg, qok, 1.0f);
    };
    const int grp1 = a.paired ? ngrp - 1 - grp0 : grp0;
    const bool ok0 = run_group(grp0), ok1 = grp1 == grp0 ? ok0 : run_group(grp1);
    if (__builtin_expect(ok0 && ok1, 1)) return;
    // (apart from the groups above and once for both: inside them it cost every call of head_dim 128 1 us, with one
    // loop around everything 5)
    int grp = ok0 ? grp1 : grp0;
#pragma clang loop unroll(disable)
    while (true) {
        __syncthreads();  // a merge before has been read
        plain_group(grp);
        if (grp == grp1 || ok1) break;
        grp = grp1;
    }
}

}  // namespace
}  // namespace dev

namespace detail {

namespace {

// positions are cut into chunks while there are fewer workgroups than this
constexpr long kMaxGroups = 256;

// QB query blocks of 32 and KS interleaved tiles per workgroup (eight waves)
struct PromptPlan {
    int qb, ks, nchunks, paired, ntiles;
    long wgs, tile_bytes, rec_bytes;
};

PromptPlan prompt_plan(int M, int H, int Hkv, int D, int kv_max) {
    PromptPlan p;
    const long nq = static_cast<long>(M) * (H / Hkv);
    auto groups = [&](int qb) { return Hkv * ((nq + 32 * qb - 1) / (32 * qb)); };
    p.qb = D > 64 || groups(4) >= 512 ? 4 : 2;
    p.ks = 8 / p.qb;
    const long g = groups(p.qb);
    p.ntiles = (kv_max + dev::kPaTile - 1) / dev::kPaTile;
    const long stages = (p.ntiles + p.ks - 1) / p.ks;
    p.nchunks = static_cast<int>(std::max<long>(1, std::min<long>({kMaxGroups / g, stages, 16})));
    p.paired = p.nchunks == 1 && g >= 512;
    p.wgs = p.paired ? Hkv * ((g / Hkv + 1) / 2) : g * p.nchunks;
    p.tile_bytes = static_cast<long>(Hkv) * p.ntiles * dev::pa_tile_bytes(D);
    p.rec_bytes = static_cast<long>(Hkv) * p.ntiles * static_cast<long>(sizeof(dev::PaTile));
    return p;
}

template <int D, int QB, int KS>
int launch_attn(const dev::PromptArgs& a, long wgs, hipStream_t stream) {
    constexpr int kMaxDevices = 64, kLds = dev::pa_lds_bytes<D, QB, KS>();
    static std::atomic<bool> ready[kMaxDevices];
    int devid = 0;
    if (hipGetDevice(&devid) != hipSuccess || devid < 0 || devid >= kMaxDevices) return kFailed;
    if (!ready[devid].load(std::memory_order_acquire)) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(&dev::prompt_attn_kernel<D, QB, KS>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, kLds) != hipSuccess)
            return kFailed;
        ready[devid].store(true, std::memory_order_release);
    }
    hipLaunchKernelGGL((dev::prompt_attn_kernel<D, QB, KS>), dim3(static_cast<unsigned>(wgs)), dim3(64 * QB * KS), kLds,
                       stream, a);
    return 0;
}

}  // namespace

bool prompt_attention_supported(int M, int head_dim) {
    return M >= kPromptAttnMinRows && (head_dim == 64 || head_dim == 128);
}

long prompt_attention_workspace_bytes(int M, int n_heads, int n_kv_heads, int head_dim, int kv_max) {
    const PromptPlan p = prompt_plan(M, n_heads, n_kv_heads, head_dim, kv_max);
    // records: M n_heads nchunks of them, and nchunks <= min(16, 256 / query groups) with at least
    // M n_heads / 128 groups; bounded so that it grows with M (a workspace sized for the longest
    // prompt serves every shorter one)
    const long recs = std::min<long>(16L * M * n_heads, kMaxGroups * 128L);
    return p.tile_bytes + p.rec_bytes + recs * (head_dim + 4) * 4;
}

// Measured (32/8 heads of 64, whole call, against the five launches per 512 rows over materialized
// scores; error: 2-norm against float64): 2048 rows 575-589 -> 70-83 us, 3.9e-7 -> 2.1e-7 (the kernel 76 us traced,
// the split 6; its MFMAs alone, in a copy without copies, softmax and maxima, 41 us over 20 us of
// launches, split, prologues and merges), 512 rows 83 -> 21 us, 512 rows at position 2000 274 -> 58 us,
// 64 rows 29 -> 14 us; heads of 128: 2048 rows 771 -> 150 us, 512 rows 110 -> 56 us.  Three bf16 parts and six
// products (exact parts, 1.1e-7 instead of 1.2e-7 at 64 rows) took 112 us at 2048 rows.  Workgroups: eight waves as 4
// blocks x 2 tiles once 512 of them exist (half the copies of 2 x 4), else 2 x 4, which fills the GPU from
// half the rows.
int launch_prompt_attention(const float* Q, long ldq, const float* K, const float* V, float* out, long ldo, int M,
                            int n_heads, int n_kv_heads, int head_dim, const int* kv_dev, int kv0, int kv_max,
                            float scale, void* ws, hipStream_t stream) {
    const int D = head_dim;
    auto a16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    if (!prompt_attention_supported(M, D) || kv_max < 1 || n_kv_heads < 1 || n_kv_heads > 65535 ||
        n_heads % n_kv_heads != 0 || ldo % 4 != 0 || !a16(out) || !a16(ws))
        return kDeclined;
    if (static_cast<long>(M) * n_heads > 0x7FFFFFFFL - 256) return kDeclined;
    const PromptPlan p = prompt_plan(M, n_heads, n_kv_heads, D, kv_max);
    if (p.wgs > 0x7FFFFFFFL) return kDeclined;
    if (p.nchunks > 1 && M > 65535) return kDeclined;  // the combine kernel's grid
    char* const base = static_cast<char*>(ws);
    dev::PaTile* const recs = reinterpret_cast<dev::PaTile*>(base + p.tile_bytes);
    dev::PromptArgs a;
    a.Q = Q;
    a.K = K;
    a.V = V;
    a.tiles = base;
    a.recs = recs;
    a.kv_dev = kv_dev;
    a.part = p.nchunks > 1 ? reinterpret_cast<float*>(base + p.tile_bytes + p.rec_bytes) : nullptr;
    a.out = p.nchunks > 1 ? nullptr : out;
    a.ldq = ldq;
    a.ldo = ldo;
    a.kv0 = kv0;
    a.M = M;
    a.G = n_heads / n_kv_heads;
    a.n_kv = n_kv_heads;
    a.ntiles = p.ntiles;
    a.nchunks = p.nchunks;
    a.paired = p.paired;
    a.qscale = scale * 1.44269504088896341f;
    const dim3 sg(static_cast<unsigned>(p.ntiles), static_cast<unsigned>(n_kv_heads));
    int rc;
    if (D == 64) {
        hipLaunchKernelGGL(dev::prompt_kv_split_kernel<64>, sg, dim3(256), 0, stream, K, V, base, recs, n_kv_heads,
                           p.ntiles, kv_dev, kv0, M);
        rc = p.qb == 4 ? launch_attn<64, 4, 2>(a, p.wgs, stream) : launch_attn<64, 2, 4>(a, p.wgs, stream);
    } else {
        hipLaunchKernelGGL(dev::prompt_kv_split_kernel<128>, sg, dim3(512), 0, stream, K, V, base, recs, n_kv_heads,
                           p.ntiles, kv_dev, kv0, M);
        rc = launch_attn<128, 4, 2>(a, p.wgs, stream);
    }
    if (rc != 0) return rc;
    if (p.nchunks > 1) launch_attention_combine(a.part, out, n_heads, M, D, p.nchunks, ldo, stream);
    return 0;
}

}  // namespace detail
}  // namespace cri
