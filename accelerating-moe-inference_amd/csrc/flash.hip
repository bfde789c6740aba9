// Causal attention in one pass per (sequence, head, tile of 128 or 256
// queries): the scores never leave the chip.
//
// Each wave owns 32 queries.  It computes the transposed scores
// S^T[key][query] = K Q^T on fp32 MFMA (32x32x2), so the accumulator column,
// i.e. the lane, is the query: every per-query quantity of the softmax (the
// running max, the denominator, the rescale) is lane-local, and the two lane
// halves, which hold different keys of the same query, meet through one
// shuffle.  The output is accumulated transposed too, O^T[dim][query] +=
// V^T P^T, with P^T fed to the MFMA straight from the score registers: the
// MFMA only needs the A and B operands to agree on which k each lane half
// supplies, so step j of the P V product takes key 8*(j/4) + 4*half + j%4,
// the key the score accumulator's register j holds, and V is read at that
// key.  No transpose through LDS, no S x S buffer in HBM.
//
// Softmax (PhiAttention::forward, src/layer.cu:118-140): score / sqrt(hd),
// keys ki <= qi within the window, weights exp(s - m); the maximum is carried
// online (rescaling the partial sums by exp(m_old - m_new)), and the output
// divides the weighted sum by the denominator at the end -- the same values
// as the reference's loop up to rounding.  The reference rounds
// float(exp(double(x))); here exp(x) is the single-precision hardware exp2 of
// x * log2(e) (relative error about |x| * 6e-8 + 1 ulp, x <= 0), which the
// online rescaling's different rounding already puts outside bit-exactness:
// the fp64 exp took about half as long as the MFMAs of a key block.  For the
// same reason the division by sqrt(hd) is folded into that multiply.
#include "common.hpp"
#include "split.hpp"

#include <cmath>

namespace moe {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kKBlock = 32;  // keys per block

// What a workgroup works on, from its place in the grid.
struct FlashTile {
    int64_t qw, kw;        // row widths of q and out, k and v
    const float *q, *k, *v;  // this sequence's first row, at this head's columns
    float* out;
    int row0;              // first query
    int S, W;              // sequence length, window (0: none); both fit 32 bits
    int k_lo, k_hi;        // keys the tile's queries can see
};

template <int HD, int NW>
__device__ __forceinline__ FlashTile flash_tile(const float* q, const float* k, const float* v,
                                                float* out, int64_t S, int64_t H, int64_t KVH,
                                                int64_t window) {
    // Causal work grows with the tile index (tile t walks 4t + 4 key blocks).
    // Workgroups half a grid apart share a CU when the grid fills two per CU
    // (the dispatcher deals ids round-robin over the XCDs and their CUs), so
    // the order is tile-major with heavy and light tiles interleaved -- rank
    // r < T/2 takes tile T-1-r, the rest tile r - T/2 -- and each CU gets a
    // heavy and a light tile (measured: 0.41 -> 0.29 ms per config-5 prefill).
    const int64_t T = gridDim.x, BH = gridDim.y;
    const int64_t L = static_cast<int64_t>(blockIdx.y) * T + blockIdx.x;
    const int64_t rank = L / BH, z = L % BH;
    // (8 waves: one workgroup per CU, heaviest first)
    const int tile = static_cast<int>(NW == 8 || rank < (T + 1) / 2 ? T - 1 - rank
                                                                    : rank - (T + 1) / 2);
    constexpr int kQTile = 32 * NW;
    const int64_t b = z / H, h = z % H, kh = h / (H / KVH);
    FlashTile t;
    t.qw = H * HD;
    t.kw = KVH * HD;
    t.q = q + b * S * t.qw + h * HD;
    t.k = k + b * S * t.kw + kh * HD;
    t.v = v + b * S * t.kw + kh * HD;
    t.out = out + b * S * t.qw + h * HD;
    t.row0 = tile * kQTile;
    t.S = static_cast<int>(S);
    t.W = static_cast<int>(window);
    t.k_hi = t.row0 + kQTile < t.S ? t.row0 + kQTile : t.S;
    t.k_lo = 0;
    if (t.W > 0 && t.row0 - (t.W - 1) > 0) t.k_lo = ((t.row0 - (t.W - 1)) / kKBlock) * kKBlock;
    return t;
}

// The online softmax of one key block's transposed scores s (this lane's
// query qi, register r = key k0 + 8*(r/4) + 4*half + r%4), replaced by their
// weights; c2 = log2(e) / sqrt(hd).  `full`: every key visible.  The running
// maximum follows the scores only once they pass it by LAG / c2, so weights
// reach 2^LAG (their ratios, all that counts, keep every bit) and the sums are
// rescaled by alpha in few blocks.  Returns whether any lane's are.  (A sum
// that only a lag overflows sends the pieces' tile to fp32 MFMA, which has none.)
template <int LAG>
__device__ __forceinline__ bool softmax_block(f32x16& s, bool full, int k0, int qi, int half,
                                               int S, int W, float c2, float& m_run, float& den,
                                               float& alpha) {
    if (!full) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int key = k0 + 8 * (r / 4) + 4 * half + (r % 4);
            const bool vis = key <= qi && key < S && (W <= 0 || qi - key < W);
            s[r] = vis ? s[r] : -INFINITY;
        }
    }
    float bmax = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) bmax = fmaxf(bmax, s[r]);
    bmax = fmaxf(bmax, __shfl_xor(bmax, 32, 64));
    // (from -inf, nothing visible yet, any visible score moves it; NaN never)
    const float m_new = LAG == 0                        ? fmaxf(m_run, bmax)
                        : (bmax - m_run) * c2 > float(LAG) ? bmax
                                                           : m_run;
    // rescale of the sums so far (none yet, or nothing visible: 1)
    alpha = m_run == -INFINITY || m_new == -INFINITY
                ? 1.0f
                : __builtin_amdgcn_exp2f((m_run - m_new) * c2);
    // a query with nothing visible yet has m_new = -inf: its masked
    // scores give weight 0
    const float mc = m_new == -INFINITY ? 0.0f : m_new * c2;
    float psum = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], c2, -mc));
        psum += s[r];
    }
    den = den * alpha + psum;
    m_run = m_new;
    return __any(alpha != 1.0f);
}

// The tile on fp32 MFMA: what the pieces below leave to it (values their
// split does not hold).  `smem`: kFp32Lds<HD> bytes.
template <int HD>
constexpr int kFp32Lds = 4 * kKBlock * (HD + 8) * 4;

template <int HD, int NW>
__device__ __forceinline__ void flash_fp32(const FlashTile& ft, float c2, unsigned char* smem) {
    static_assert(HD % 32 == 0 && HD <= 128, "head_dim 32, 64, 96 or 128");
    constexpr int LD = HD + 8;      // LDS row stride: the lane halves land 32 banks apart
    constexpr int QK = HD / 2;      // MFMA steps of the score product (2 dims each)
    constexpr int MB = HD / 32;     // 32-dim blocks of the output
    // two K/V buffers: block j is staged into buffer j % 2 while the waves
    // read block j - 1 from the other, so one barrier per block suffices
    auto Ks = reinterpret_cast<float(*)[kKBlock * LD]>(smem);
    auto Vs = Ks + 2;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: scalar branches
    const int lq = lane & 31, half = lane >> 5;
    const int64_t kw = ft.kw;
    const int S32 = ft.S, W = ft.W, k_lo = ft.k_lo, k_hi = ft.k_hi;
    const int q0 = ft.row0 + 32 * wave;               // this wave's first query
    const int qi = q0 + lq;                           // this lane's query
    const bool wave_live = q0 < S32;
    const float *kb = ft.k, *vb = ft.v;

    // Q^T operand: step j, half h supplies dim h*QK + j of this lane's query
    float qr[QK];
    {
        const float* qrow = ft.q + (qi < S32 ? qi : S32 - 1) * ft.qw + half * QK;
#pragma unroll
        for (int j = 0; j < QK; j += 4) {
            const f32x4 t = *reinterpret_cast<const f32x4*>(qrow + j);
            qr[j] = t[0];
            qr[j + 1] = t[1];
            qr[j + 2] = t[2];
            qr[j + 3] = t[3];
        }
    }

    // block staging: 32 keys x HD floats of K and of V, 16-byte chunks
    constexpr int CHUNKS = kKBlock * HD / 4;       // per matrix
    constexpr int PER_T = (CHUNKS + 64 * NW - 1) / (64 * NW);
    f32x4 kst[PER_T], vst[PER_T];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < PER_T; ++i) {
            const int c = tid + 64 * NW * i;
            if (c < CHUNKS) {
                const int r = c / (HD / 4), col = 4 * (c % (HD / 4));
                int key = k0 + r;
                key = key < S32 ? key : S32 - 1;  // past the end: a valid row, masked below
                kst[i] = *reinterpret_cast<const f32x4*>(kb + key * kw + col);
                vst[i] = *reinterpret_cast<const f32x4*>(vb + key * kw + col);
            }
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < PER_T; ++i) {
            const int c = tid + 64 * NW * i;
            if (c < CHUNKS) {
                const int r = c / (HD / 4), col = 4 * (c % (HD / 4));
                *reinterpret_cast<f32x4*>(&Ks[buf][r * LD + col]) = kst[i];
                *reinterpret_cast<f32x4*>(&Vs[buf][r * LD + col]) = vst[i];
            }
        }
    };

    f32x16 acc[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][r] = 0.0f;
    float m_run = -INFINITY, den = 0.0f;
    const int wq_last = q0 + 31 < S32 ? q0 + 31 : S32 - 1;  // the wave's last query

    fetch(k_lo);
    stage(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = k_lo; k0 < k_hi; k0 += kKBlock) {
        const bool more = k0 + kKBlock < k_hi;
        if (more) fetch(k0 + kKBlock);
        // the wave skips blocks wholly after its last query or before its
        // first query's window (wave-uniform)
        bool active = wave_live && k0 <= wq_last;
        if (W > 0 && k0 + kKBlock - 1 < q0 - (W - 1)) active = false;
        if (active) {
            // S^T = K Q^T: lane = query, register r = key 8*(r/4) + 4*half + r%4
            f32x16 s;
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 0.0f;
            const float* krow = &Ks[buf][lq * LD + half * QK];
#pragma unroll
            for (int j = 0; j < QK; j += 4) {
                const f32x4 kk = *reinterpret_cast<const f32x4*>(krow + j);
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(kk[t], qr[j + t], s, 0, 0, 0);
            }
            // every key of the block visible to every query of the wave:
            // no mask (wave-uniform)
            const bool full = k0 + kKBlock - 1 <= q0 && (W <= 0 || wq_last - k0 < W);
            float alpha;
            if (softmax_block<0>(s, full, k0, qi, half, S32, W, c2, m_run, den, alpha)) {
#pragma unroll
                for (int m = 0; m < MB; ++m)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[m][r] *= alpha;
            }
            // O^T += V^T P^T: step j takes key 8*(j/4) + 4*half + j%4
            const float* vcol = &Vs[buf][lq];
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int key = 8 * (j / 4) + 4 * half + (j % 4);
#pragma unroll
                for (int m = 0; m < MB; ++m)
                    acc[m] = __builtin_amdgcn_mfma_f32_32x32x2f32(vcol[key * LD + 32 * m], s[j],
                                                                  acc[m], 0, 0, 0);
            }
        }
        if (more) stage(buf ^ 1);  // the other buffer's last readers passed the previous barrier
        __syncthreads();
        buf ^= 1;
    }

    // out[query][dim] = O^T[dim][query] / den; register r of block m is dim
    // 32m + 8*(r/4) + 4*half + r%4: four consecutive dims per group
    const float den_all = den + __shfl_xor(den, 32, 64);
    if (wave_live && qi < S32) {
        float* orow = ft.out + qi * ft.qw;
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                f32x4 o;
#pragma unroll
                for (int t = 0; t < 4; ++t) o[t] = acc[m][4 * g + t] / den_all;
                *reinterpret_cast<f32x4*>(orow + 32 * m + 8 * g + 4 * half) = o;
            }
    }
}

// The tile on the bf16 pieces (split.hpp): keys and values are split once per
// workgroup on their way to LDS, the queries once into registers, the softmax
// weights (lane-local, as above) in registers; S^T = K Q^T and O^T += V^T P^T
// run on v_mfma_f32_32x32x16_bf16, six per 16 dims or keys.
//
// K planes: per piece, 16-dim chunk and half of it, 32 keys of 16 bytes (8
// dims, one lane's operand).  V planes are transposed: per piece, 16-key chunk
// c and lane half h, HD dims of 16 bytes, the 8 keys 16c + 8*(j/4) + 4h + j%4
// that registers 8c .. 8c+7 of the scores hold in that half, so P^T again goes
// to the MFMA as it comes.  A thread takes 4 keys of two adjacent dims (the
// even one in the first 32 slots of 64 dims, the odd one in the next 32, so
// neighbouring lanes store side by side): accumulator block 2b + e, row i is
// dim 64b + 2i + e.  The next block's rows are in flight in registers while a
// block is computed.  Four waves keep one stage of planes (26 KB at head_dim
// 64), written between two barriers while the CU's other workgroup computes;
// eight keep two (101 KB at head_dim 128).
//
// Bound: the waves' own chain, scores -> softmax -> weights -> output; at
// head_dim 128 a wave's block is 96 MFMAs (3,072 cycles) and about 390 vector
// instructions (1,560), and two waves share a SIMD.  Measured on MI355X, fp32
// MFMA -> here: 2 x 2047 queries, 32 heads of 128, 689 -> 359 us (100 -> 192
// TFLOP/s); 4 x 2048, 16 heads, window 512, 366 -> 230; 2 x 2048, 32 heads of
// 64, 315 -> 187; 8 x 512, 16 heads of 64, 54.4 -> 48.2.  Error against 64 bits
// 3.1e-7 -> 2.6e-7, 2.9e-7 -> 2.4e-7, 3.0e-7 -> 2.5e-7, 1.8e-7 -> 1.5e-7.  The lagging
// maximum took the first from 516 to 505 us on four waves, eight waves to 377, a
// split without a look for small values to 359.
//
// The pieces hold every query, key, value and weight below 2^105 exactly, so
// the scores and the outputs' sums carry the scale 2^46 (split.hpp): c2 and the
// last division take it out.
template <int HD>
struct FlashPlanes {
    static constexpr int KH = kKBlock * 16 + 16;  // bytes of a K half plane
    static constexpr int VH = HD * 16 + 64;       // ... of a V one
    static constexpr int V0 = 3 * (HD / 16) * 2 * KH;
    static constexpr int BYTES = V0 + 12 * VH;
    static __device__ __forceinline__ int k_at(int piece, int ch, int half, int key) {
        return ((piece * (HD / 16) + ch) * 2 + half) * KH + key * 16;
    }
    static __device__ __forceinline__ int v_at(int piece, int c, int half, int slot) {
        return V0 + ((piece * 2 + c) * 2 + half) * VH + slot * 16;
    }
};

// Returns whether the tile's sums came out finite, every value of it split
// exactly; the output is written only then.
template <int HD, int NW>
__device__ __forceinline__ bool flash_pieces(const FlashTile& ft, float c2, unsigned char* smem) {
    constexpr int T = 64 * NW;
    constexpr int NBUF = NW == 8 ? 2 : 1;  // stages of planes
    using PL = FlashPlanes<HD>;
    constexpr int CH = HD / 16;   // 16-dim chunks
    constexpr int MB = HD / 32;   // 32-dim blocks of the output
    constexpr int KC = kKBlock * HD / 4 / T;  // 16-byte chunks of K per thread
    // 4-key x 2-dim blocks of V per thread; where there are fewer of them than
    // threads, the first VN threads (whole waves) take one each
    constexpr int VN = kKBlock * HD / 8, VC = VN >= T ? VN / T : 1;
    auto v_mine = [&](int c) { return VN >= T || c < VN; };
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lq = lane & 31, half = lane >> 5;
    const int S = ft.S, W = ft.W;
    const int q0 = ft.row0 + 32 * wave, qi = q0 + lq;
    const bool wave_live = q0 < S;
    const int wq_last = q0 + 31 < S ? q0 + 31 : S - 1;

    // Q^T operand of chunk ch: dims 16 ch + 8 half .. + 7 of this lane's query
    const float* qrow = ft.q + (qi < S ? qi : S - 1) * ft.qw + 8 * half;
    u32x4 qp[CH][3];
#pragma unroll
    for (int ch = 0; ch < CH; ++ch)
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const f32x2 x = *reinterpret_cast<const f32x2*>(qrow + 16 * ch + 2 * p);
            uint32_t w[3];
            split_pair(x[0], x[1], w);
#pragma unroll
            for (int t = 0; t < 3; ++t) qp[ch][t][p] = w[t];
        }

    f32x4 kst[KC];
    f32x2 vst[VC][4];
    // rows k0 .. k0 + 31 from wave-uniform bases, 32-bit lane offsets; keys past
    // the end: the last row, masked
    const uint32_t kw4 = static_cast<uint32_t>(ft.kw) * 4;
    auto fetch = [&](int k0) {
        const char* kb = reinterpret_cast<const char*>(ft.k + static_cast<int64_t>(k0) * ft.kw);
        const char* vb = reinterpret_cast<const char*>(ft.v + static_cast<int64_t>(k0) * ft.kw);
        const int lim = S - 1 - k0;
        auto row = [&](int r) { return static_cast<uint32_t>(r < lim ? r : lim) * kw4; };
#pragma unroll
        for (int i = 0; i < KC; ++i) {
            const int c = tid + T * i;
            kst[i] = *reinterpret_cast<const f32x4*>(kb + (row(c / (HD / 4)) + 16 * (c % (HD / 4))));
        }
#pragma unroll
        for (int i = 0; i < VC; ++i) {
            const int c = tid + T * i;
            if (!v_mine(c)) break;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                vst[i][j] = *reinterpret_cast<const f32x2*>(
                    vb + (row(4 * (c / (HD / 2)) + j) + 8 * (c % (HD / 2))));
        }
    };
    auto store4 = [&](const f32x4& x, unsigned char* at, int plane) {
        uint32_t a[3], b[3];
        split_pair(x[0], x[1], a);
        split_pair(x[2], x[3], b);
#pragma unroll
        for (int t = 0; t < 3; ++t) *reinterpret_cast<u32x2*>(at + t * plane) = u32x2{a[t], b[t]};
    };
    auto stage = [&](unsigned char* to) {
#pragma unroll
        for (int i = 0; i < KC; ++i) {
            const int c = tid + T * i, key = c / (HD / 4), col = 4 * (c % (HD / 4));
            store4(kst[i], to + PL::k_at(0, col / 16, (col / 8) & 1, key) + (col & 4) * 2, CH * 2 * PL::KH);
        }
#pragma unroll
        for (int i = 0; i < VC; ++i) {
            const int c = tid + T * i, kg = c / (HD / 2), dp = c % (HD / 2);
            if (!v_mine(c)) break;
            const int slot = (dp & ~31) * 2 + (dp & 31);
#pragma unroll
            for (int e = 0; e < 2; ++e)
                store4(f32x4{vst[i][0][e], vst[i][1][e], vst[i][2][e], vst[i][3][e]},
                       to + PL::v_at(0, kg / 4, kg & 1, slot + 32 * e) + (kg & 2) * 4, 4 * PL::VH);
        }
    };
    const unsigned char* cur = smem;
    auto frag = [&](int at) {
        return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(cur + at));
    };

    f32x16 acc[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][r] = 0.0f;
    float m_run = -INFINITY, den = 0.0f;

    fetch(ft.k_lo);
    for (int k0 = ft.k_lo; k0 < ft.k_hi; k0 += kKBlock) {
        // one stage: the previous block's planes have been read; two: the ones
        // written now were read before the previous block's barrier
        if (NBUF == 1) __syncthreads();
        unsigned char* to = smem + (NBUF == 2 && ((k0 / kKBlock) & 1) ? PL::BYTES : 0);
        stage(to);
        __syncthreads();
        cur = to;
        if (k0 + kKBlock < ft.k_hi) fetch(k0 + kKBlock);
        bool active = wave_live && k0 <= wq_last;
        if (W > 0 && k0 + kKBlock - 1 < q0 - (W - 1)) active = false;
        if (!active) continue;
        f32x16 s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.0f;
#pragma unroll
        for (int ch = 0; ch < CH; ++ch) {
            bf16x8 kp[3];
#pragma unroll
            for (int t = 0; t < 3; ++t) kp[t] = frag(PL::k_at(t, ch, half, lq));
#pragma unroll
            for (int t = 0; t < kSplitTerms; ++t)
                s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    kp[kSplitA[t]], __builtin_bit_cast(bf16x8, qp[ch][kSplitB[t]]), s, 0, 0, 0);
        }
        const bool full = k0 + kKBlock - 1 <= q0 && (W <= 0 || wq_last - k0 < W);
        float alpha;
        if (softmax_block<8>(s, full, k0, qi, half, S, W, c2 * kSplitUnscale, m_run, den, alpha)) {
#pragma unroll
            for (int m = 0; m < MB; ++m)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[m][r] *= alpha;
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            u32x4 pp[3];
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                uint32_t w[3];
                split_pair(s[8 * c + 2 * p], s[8 * c + 2 * p + 1], w);
#pragma unroll
                for (int t = 0; t < 3; ++t) pp[t][p] = w[t];
            }
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                bf16x8 vp[3];
#pragma unroll
                for (int t = 0; t < 3; ++t) vp[t] = frag(PL::v_at(t, c, half, 32 * m + lq));
#pragma unroll
                for (int t = 0; t < kSplitTerms; ++t)
                    acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        vp[kSplitA[t]], __builtin_bit_cast(bf16x8, pp[kSplitB[t]]), acc[m], 0, 0, 0);
            }
        }
    }

    // What the pieces do not hold: non-finite sums, and queries whose scores all
    // passed the range (every query sees a key, so a sum of weights is above 0)
    const float den_all = den + __shfl_xor(den, 32, 64);
    int bad = 0;
    if (wave_live && qi < S) {
        float z = den_all * 0.0f;
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int r = 0; r < 16; ++r) z = fmaf(acc[m][r], 0.0f, z);
        bad = !(z == 0.0f && den_all > 0.0f);
    }
    if (__syncthreads_or(bad)) return false;

    if (wave_live && qi < S) {
        const float den_s = den_all / kSplitUnscale;
        float* orow = ft.out + qi * ft.qw;
#pragma unroll
        for (int b = 0; b < MB / 2; ++b)
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    // dims 64b + 2i, + 1 of rows i = 8g + 4 half + 2u, + 1
                    const int r = 4 * g + 2 * u;
                    f32x4 o{acc[2 * b][r], acc[2 * b + 1][r], acc[2 * b][r + 1],
                            acc[2 * b + 1][r + 1]};
#pragma unroll
                    for (int t = 0; t < 4; ++t) o[t] = o[t] / den_s;
                    *reinterpret_cast<f32x4*>(orow + 64 * b + 16 * g + 8 * half + 4 * u) = o;
                }
    }
    return true;
}

// At least two waves per SIMD: at most 256 registers a lane.
template <int HD, int NW, bool PIECES>
__global__ __launch_bounds__(64 * NW, 2) void flash_attn_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    float* __restrict__ out, int64_t S, int64_t H, int64_t KVH, int64_t window, float scale) {
    static_assert(HD == 64 || HD == 128, "head_dim 64 or 128");
    constexpr int PLANES = PIECES ? FlashPlanes<HD>::BYTES * (NW == 8 ? 2 : 1) : 0;
    constexpr int LDS = PLANES > kFp32Lds<HD> ? PLANES : kFp32Lds<HD>;
    __shared__ __align__(16) unsigned char smem[LDS];
    const FlashTile ft = flash_tile<HD, NW>(q, k, v, out, S, H, KVH, window);
    // the running maximum is kept on the unscaled scores: s / scale is
    // monotone in s, so exp(s/scale - m/scale) = exp2((s - m) * c) with
    // c = log2(e) / scale, one multiply per weight instead of a division
    const float c2 = 1.44269504088896340736f / scale;
    if constexpr (PIECES) {
        if (flash_pieces<HD, NW>(ft, c2, smem)) return;
    }
    flash_fp32<HD, NW>(ft, c2, smem);
}

}  // namespace

bool launch_flash_attention(const float* q, const float* k, const float* v, float* out,
                            int64_t batch, int64_t seq_len, int64_t q_heads, int64_t kv_heads,
                            int64_t head_dim, int64_t window, hipStream_t s) {
    if (seq_len > INT32_MAX) return false;  // key indices are 32-bit
    const float scale = sqrtf(static_cast<float>(head_dim));
    auto run = [&](auto kernel, int waves) {
        const dim3 grid(static_cast<unsigned>(ceil_div(seq_len, 32 * waves)),
                        static_cast<unsigned>(batch * q_heads));
        hipLaunchKernelGGL(kernel, grid, dim3(64 * waves), 0, s, q, k, v, out, seq_len, q_heads,
                           kv_heads, window, scale);
    };
    // Four waves, two workgroups per CU, or eight waves with two stages of
    // planes, which stage half as much per wave and meet once per block but
    // balance the causal tiles less finely, and whose 256-query tiles walk blocks
    // that a short sequence or window hides from most of their waves.  us on
    // MI355X, fp32 MFMA / four / eight waves: head_dim 64, 512 tiles of 128 queries
    // 54.4 / 41.2 / 52.6; 1,024 tiles and more, 2,048 keys 313 / 201 / 191, 1,396 keys
    // 604 / 388 / 453, 100 keys 83 / 57 / 98, windows of 16 / 64 / 256 / 1,024 of 1,396
    // keys 122 / 83 / 146, 145 / 95 / 156, 268 / 166 / 229, 547 / 360 / 393; head_dim 128
    // (fp32 MFMA / eight waves), 512 tiles 97 / 76, 1,024 tiles 689 / 344, there with a
    // window of 16 100 / 83.  Up to 256 tiles of head_dim 128, at most one workgroup per
    // CU, are bound by one wave's chain through its key blocks, which the splits
    // lengthen: 81 / 85 (four) / 85 and 46.6 / 51 / 49.8.
    const int64_t tiles = ceil_div(seq_len, 128) * batch * q_heads;
    const int64_t keys = window > 0 && window < seq_len ? window : seq_len;
    switch (head_dim) {
        case 64:
            if (tiles >= 1024 && keys > 1536) run(flash_attn_kernel<64, 8, true>, 8);
            else run(flash_attn_kernel<64, 4, true>, 4);
            return true;
        case 128:
            if (tiles >= 512) run(flash_attn_kernel<128, 8, true>, 8);
            else run(flash_attn_kernel<128, 4, false>, 4);
            return true;
        default:
            return false;
    }
}

}  // namespace moe
