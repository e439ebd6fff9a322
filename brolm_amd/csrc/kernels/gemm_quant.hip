// Linear on quantized weights for 17 rows and more, on MFMA: Y[M,N] = X[M,K]
// deq(W)[N,K]^T with the weights rounded once to FP16 (FP32 multiply-add, one
// rounding), FP32 accumulation.  K a multiple of 256.
//
// A workgroup of eight wavefronts computes a (32 FM) x (128 FN) tile over a K
// slice.  Wavefronts w and w + 4 share the columns 32 w .. 32 w + 31 of each of
// the FN groups of 128 and take every second 64-element unit of K, so no
// weight is decoded twice in a workgroup and every SIMD has two wavefronts, one
// decoding while the other multiplies.  Both operands come by LDS-DMA:
//   A   stages of 128 K elements, NA slots, shared by all wavefronts (one
//       barrier a stage); 16-byte chunks XOR-swizzled by the row
//   W   the raw quantized bytes, NB blocks deep; a lane reads the bytes of its
//       own MFMA column and decodes them into the B operand's registers.  A
//       decoded value never passes through LDS.
// The K elements of one MFMA are the ones a lane's 16 bytes hold (see Fmt);
// the A reads follow that order.
//
// The epilogue goes through LDS (the two wavefronts' sums added in a fixed
// order) and a compact row loop: unrolled over the accumulators it was
// thousands of instructions run once, and their fetches cost more than the
// arithmetic (a 128 x 128 tile's fixed time 17 us, of 24 at K = 2048).
//
// What bounds it: no unit alone.  The decode (about three instructions a weight)
// and the MFMAs of a wavefront alternate, and the two wavefronts of a SIMD cover
// each other in part: VALU busy 45 to 52 %, MFMA 15 to 24 %, LDS active 12 to 17 %
// (75 and 300 rows), with a third of the wave cycles waiting: the fill, the ring's
// barriers, the exchange of partials.  Measured against the tile kernels of
// gemm.hip that ran these shapes before (one launch, weights from HBM):
// 75 x 6144 x 2048 Q4_K 44.2 -> 13.6 us, 300 x 2048 x 6144 Q6_K 98 -> 25.3 us,
// 2000 x 6144 x 2048 Q4_K 94 -> 79 us, SwiGLU 128 x 3072 x 1024 Q4_K 14.1 -> 7.9.
//
// Where the tiles leave CUs idle, S workgroups share a tile's K: each writes
// its FP32 partials by device-scope stores to the linear workspace, the last
// to arrive (tagged_arrive) adds the S partials in slice order and runs the
// epilogue, so the result does not depend on the order of arrival.
#include <algorithm>

#include "carrier_layout.h"
#include "gemm_job.h"

namespace bx {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));

constexpr int kThreads = 512;

struct QuantJob {
    TileJob t;
    int S;              // K slices
    uint64_t* cnt;      // S > 1: arrival counters, FP32 partials, launch tag
    float* part;
    uint32_t tag;
};

// Two small unsigned integers v at bits 0 and 16, as an FP16 pair: left alone
// they are the subnormals v 2^-24, and OR-ed with kMagic the numbers 1024 + v.
constexpr uint32_t kMagic = 0x64006400u;
constexpr float kSub = 16777216.f;   // 2^24
// f16(h * d + c) of the low or the high half of a pair: one FP32 multiply-add
// and one rounding (v_fma_mixlo / mixhi).  Every product and every c below is
// exact in FP32 (11-bit d, scales of 6 or 8 bits), so the weights have the bits
// of bx_dequant_to_f16.  Q4_K takes the subnormals, with d 2^24: its c is then
// the minimum alone, where -1024 d - min would be rounded, to as much as 2^-14
// of a quantization step (0.04 % of the weights one FP16 value off, and a zero
// weight 6e-5 d).  Same instructions, same time (75 x 6144 x 2048).
__device__ __forceinline__ _Float16 mad_lo(uint32_t v, float d, float c) {
    return (_Float16)__builtin_fmaf((float)as_h2(v).x, d, c);
}
__device__ __forceinline__ _Float16 mad_hi(uint32_t v, float d, float c) {
    return (_Float16)__builtin_fmaf((float)as_h2(v).y, d, c);
}
// eight weights in K order from the pairs (e0 e2), (e1 e3), (e4 e6), (e5 e7)
__device__ __forceinline__ h8 weights8(uint32_t p02, uint32_t p13, uint32_t p46, uint32_t p57, float d, float c) {
    return h8{mad_lo(p02, d, c), mad_lo(p13, d, c), mad_hi(p02, d, c), mad_hi(p13, d, c),
              mad_lo(p46, d, c), mad_lo(p57, d, c), mad_hi(p46, d, c), mad_hi(p57, d, c)};
}
// (v & mask) | or_ as one instruction: the magic sits in a vector register
// (an instruction reads one literal at most), the mask in a scalar one
__device__ __forceinline__ uint32_t bits(uint32_t v, uint32_t mask, uint32_t or_) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(mask), "v"(or_));
    return r;
}

// Per format, for 32 columns (lane: column l % 32, half lh = l / 32), a unit
// of 64 K elements (two per 128-element half h of a 256-block) in four MFMA
// steps of 16; step s multiplies the eight elements from 8 * chunk8(u, s, lh)
// of the half.
//   kHalf   copies per wavefront and 32 columns for a half, kBlk for a block
//           (the other wavefront of the pair copies the other half of them),
//           kScale for the scales of 64 columns (both copy them)
//   bytes   LDS per wavefront pair and buffer
template <int FMT>
struct Fmt;

template <>
struct Fmt<BX_TYPE_Q4_K> {
    static constexpr int kHalf = 0, kBlk = 2, kScale = 1;
    static constexpr int half_bytes(int) { return 0; }
    static constexpr int blk_bytes(int fn) { return 32 * fn * 128 + 1024; }
    static constexpr int chunk8(int u, int s) { return 8 * u + 4 * (s >> 1) + (s & 1); }
    static constexpr int lh_chunk(int lh) { return 2 * lh; }
    struct Scale { u4v h; };
    struct Raw { u4v q; };
};
template <>
struct Fmt<BX_TYPE_Q6_K> {
    static constexpr int kHalf = 0, kBlk = 3, kScale = 2;
    static constexpr int half_bytes(int) { return 0; }
    static constexpr int blk_bytes(int fn) { return 32 * fn * 192 + 1024 + 256; }
    static constexpr int chunk8(int u, int s) { return 4 * s + 2 * u; }
    static constexpr int lh_chunk(int lh) { return lh; }
    struct Scale { u4v sc; uint32_t d; };
    struct Raw { u4v ql; u2v qh; };
};
template <>
struct Fmt<BX_TYPE_Q8_0> {
    static constexpr int kHalf = 2, kBlk = 0, kScale = 1;
    static constexpr int half_bytes(int fn) { return 32 * fn * 128; }
    static constexpr int blk_bytes(int) { return 1024; }
    static constexpr int chunk8(int u, int s) { return 8 * u + 4 * (s >> 1) + (s & 1); }
    static constexpr int lh_chunk(int lh) { return 2 * lh; }
    struct Scale { u4v d; };
    struct Raw { u4v q[2]; };
};

// LDS plan of one instantiation: NA slots of A, NH half and NB block buffers
// of raw weights per wavefront pair, as deep as 160 KB allow.
template <int FMT, int FM, int FN>
struct QShape {
    using F = Fmt<FMT>;
    static constexpr int BM = 32 * FM, BN = 128 * FN;
    static constexpr int PA = BM / 32;                            // A copies per wavefront and stage,
    static constexpr int PH = F::kHalf * FN;                      // weight copies per half
    static constexpr int PB = F::kBlk * FN + F::kScale;           // and per block
    static constexpr int kSlot = BM * 256;                        // bytes of one A stage
    static constexpr int kMax = 160 * 1024 - 64;
    static constexpr int wave_bytes(int nh, int nbk) { return nh * F::half_bytes(FN) + nbk * F::blk_bytes(FN); }
    static constexpr bool fits(int na, int nh, int nbk) { return na * kSlot + 4 * wave_bytes(nh, nbk) <= kMax; }
    static constexpr int NH = F::kHalf == 0 ? 1 : fits(2, 3, 2) ? 3 : 2;
    static constexpr int NB = F::kHalf != 0 ? 2 : fits(3, NH, 3) ? 3 : 2;
    static constexpr int NA = fits(4, NH, NB) ? 4 : fits(3, NH, NB) ? 3 : 2;
    static constexpr int kWave = wave_bytes(NH, NB);
    static constexpr int kRow = BN * 4 + 16;                      // epilogue: bytes of a staged FP32 row
    static constexpr int kLds = NA * kSlot + 4 * kWave > BM * kRow ? NA * kSlot + 4 * kWave : BM * kRow;
    static_assert(fits(NA, NH, NB) && kLds <= kMax, "tile stages exceed the LDS");

    // Step H of the K loop (a half) first waits, then issues, in this order,
    // A(H + NA - 1), half(H + NH - 1) and, at even H, block(H / 2 + NB - 1).
    // The copies a wavefront issued after the ones half H needs may stay in
    // flight at its wait: counted backwards from the newest.
    static constexpr int fly(int h) {
        const int H = 64 + h;
        int n = 0;
        for (int v = H - 1;; --v) {
            if (v % 2 == 0) {
                if (v / 2 + NB - 1 == H / 2) return n;
                n += PB;
            }
            if (PH > 0) {
                if (v + NH - 1 == H) return n;
                n += PH;
            }
            if (v + NA - 1 == H) return n;
            n += PA;
        }
    }
    static constexpr int kFirst = -2 * (NA + NH + NB);   // the loop's issues before step 0, from here
};

// The four B fragments (steps s) of unit u of half h from the lane's raw bytes.
__device__ __forceinline__ void decode(const Fmt<BX_TYPE_Q4_K>::Raw& r, const Fmt<BX_TYPE_Q4_K>::Scale& sc, int h, int u,
                                       h8 (&b)[4]) {
    const float d = h2f(sc.h.x & 0xffff), dmin = h2f(sc.h.x >> 16);
    int s0, m0, s1, m1;
    q4k_pair_scales(sc.h.y, sc.h.z, sc.h.w, 2 * h + u, s0, m0, s1, m1);
    // low nibbles: q 2^-24; high nibbles, left in place: 16 q 2^-24
    const float dl = d * kSub * (float)s0, dh = d * (kSub * 0.0625f) * (float)s1;
    const float cl = -(dmin * (float)m0), ch = -(dmin * (float)m1);
    const uint32_t w[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const uint32_t x = w[2 * p], y = w[2 * p + 1], x8 = x >> 8, y8 = y >> 8;
        b[p] = weights8(x & 0x000F000Fu, x8 & 0x000F000Fu, y & 0x000F000Fu, y8 & 0x000F000Fu, dl, cl);
        b[2 + p] = weights8(x & 0x00F000F0u, x8 & 0x00F000F0u, y & 0x00F000F0u, y8 & 0x00F000F0u, dh, ch);
    }
}
__device__ __forceinline__ void decode(const Fmt<BX_TYPE_Q6_K>::Raw& r, const Fmt<BX_TYPE_Q6_K>::Scale& sc, int h, int u,
                                       h8 (&b)[4]) {
    const float d = h2f((uint16_t)sc.d);
    // the half's eight scales: steps 0, 1 in the first dword, 2, 3 in the second
    const uint32_t sw[2] = {h ? sc.sc.z : sc.sc.x, h ? sc.sc.w : sc.sc.y};
    const uint32_t lo[2] = {r.ql.x, r.ql.y}, hi[2] = {r.ql.z, r.ql.w}, qh[2] = {r.qh.x, r.qh.y};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        // low nibbles 1024 + q, high nibbles in place 1024 + 16 q (q = 0 .. 63, value q - 32)
        const float sv = (float)(int8_t)(sw[s >> 1] >> (16 * (s & 1) + 8 * u)) * d * (s < 2 ? 1.f : 0.0625f);
        const float c = sv * (s < 2 ? -1056.f : -1536.f);
        uint32_t p[4];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint32_t n = (s & 1) ? hi[j] : lo[j], q = qh[j];
            const uint32_t nm = s < 2 ? 0x000F000Fu : 0x00F000F0u, qm = s < 2 ? 0x00300030u : 0x03000300u;
            // the two high bits of step s sit at bits 2 s of each byte; they go to bits 4 (low) or 8 (in place)
            const uint32_t e = (s & 1) ? q << 2 : q << 4, o = (s & 1) ? q >> 6 : q >> 4;
            p[2 * j] = bits(e, qm, bits(n, nm, kMagic));
            p[2 * j + 1] = bits(o, qm, bits(n >> 8, nm, kMagic));
        }
        b[s] = weights8(p[0], p[1], p[2], p[3], sv, c);
    }
}
__device__ __forceinline__ void decode(const Fmt<BX_TYPE_Q8_0>::Raw& r, const Fmt<BX_TYPE_Q8_0>::Scale& sc, int h, int u,
                                       h8 (&b)[4]) {
    // blocks 4 h + 2 u and + 1 of the eight: one dword of two FP16 scales
    const uint32_t dw = h ? (u ? sc.d.w : sc.d.z) : (u ? sc.d.y : sc.d.x);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const float d = h2f((uint16_t)(dw >> (16 * p))), c = -1152.f * d;
        const uint32_t w[4] = {r.q[p].x ^ 0x80808080u, r.q[p].y ^ 0x80808080u, r.q[p].z ^ 0x80808080u,
                               r.q[p].w ^ 0x80808080u};
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint32_t x = w[2 * q], y = w[2 * q + 1];
            b[2 * p + q] = weights8(bits(x, 0x00FF00FFu, kMagic), bits(x >> 8, 0x00FF00FFu, kMagic),
                                    bits(y, 0x00FF00FFu, kMagic), bits(y >> 8, 0x00FF00FFu, kMagic), d, c);
        }
    }
}

// Four consecutive FP16 outputs, one 8-byte store where the address allows.
__device__ __forceinline__ void store4(uint16_t* p, const uint16_t (&o)[4], bool vec, int left) {
    if (vec && (reinterpret_cast<uintptr_t>(p) & 7) == 0) {
        *reinterpret_cast<u2v*>(p) = u2v{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
        return;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (k < left) p[k] = o[k];
}

template <int FMT, int FM, int FN>
__global__ __launch_bounds__(kThreads, 1) void gemm_quant_kernel(QuantJob job, const uint16_t* __restrict__ X,
                                                           const uint16_t* __restrict__ bias, int M, int K, int epi) {
    using F = Fmt<FMT>;
    using Sh = QShape<FMT, FM, FN>;
    constexpr int BM = Sh::BM, BN = Sh::BN, R = 32 * FN, NA = Sh::NA, PA = Sh::PA;
    extern __shared__ __align__(1024) unsigned char smem[];
    __shared__ uint32_t last;
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave = wid & 3, u = wid >> 2;   // columns, K units
    const int lr = lane & 31, lh = lane >> 5;

    // block -> (column tile, K slice, row tile), row tiles fastest
    int tiles = 0;
    for (int i = 0; i < job.t.members; ++i) tiles += job.t.tiles_n[i];
    const int S = job.S;
    const int idx = xcd_tile((int)blockIdx.x, job.t.tiles_m * tiles * S);
    const int tm = idx % job.t.tiles_m, rest = idx / job.t.tiles_m;
    const int s = rest % S;
    int tn = rest / S;
    const int tile = tn * job.t.tiles_m + tm;
    int mem = 0;
    while (tn >= job.t.tiles_n[mem]) tn -= job.t.tiles_n[mem++];
    // SwiGLU tiles: gate in the first half of the columns, up in the second (FN 2:
    // column groups 0 and 1 of a wavefront, FN 1: wavefronts 0, 1 and 2, 3)
    const bool two = epi == EPI_SWIGLU;
    const int N = job.t.N[mem];
    const int m0 = tm * BM, n0 = tn * (two ? BN / 2 : BN);
    const int nb = K / 256;
    const int b0 = s * nb / S, nblk = (s + 1) * nb / S - b0;   // >= 1
    const int nh = 2 * nblk;
    // first column of this wavefront in group g
    auto col0 = [&](int g) { return n0 + (two ? 32 * (FN == 2 ? wave : wave & 1) : 32 * wave + 128 * g); };
    auto weight = [&](int g) {
        return static_cast<const unsigned char*>(two ? job.t.W[FN == 2 ? g : wave >> 1] : job.t.W[mem]);
    };

    const uint32_t lbase = lds_addr(smem);
    unsigned char* const raw = smem + NA * Sh::kSlot + wave * Sh::kWave;
    const uint32_t rbase = lbase + NA * Sh::kSlot + wave * Sh::kWave;

    // ---- sources of the copies
    uint32_t va[PA];
#pragma unroll
    for (int j = 0; j < PA; ++j) {
        const int r = 4 * (wid * PA + j) + (lane >> 4);
        va[j] = (uint32_t)(min(m0 + r, M - 1) - m0) * (uint32_t)K * 2u + (uint32_t)(((lane & 15) ^ (r & 15)) * 16);
    }
    const unsigned char* const xb = reinterpret_cast<const unsigned char*>(X + (int64_t)m0 * K) + (int64_t)b0 * 512;
    // 128-byte rows (Q4_K qs, Q6_K ql: one block; Q8_0: one half), eight rows a copy
    constexpr int kRowBlk = FMT == BX_TYPE_Q8_0 ? 256 : 128;   // bytes of a row's block
    uint32_t vq[2 * FN], vh[FMT == BX_TYPE_Q6_K ? FN : 1];
    const unsigned char* qb[FN];
    const unsigned char* hb[FN];
    const unsigned char* scp[2];   // this lane's scale streams
#pragma unroll
    for (int g = 0; g < FN; ++g) {
        const int c0 = min(col0(g), N - 1);
        qb[g] = weight(g) + (int64_t)c0 * nb * kRowBlk + (int64_t)b0 * kRowBlk;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int r = 16 * u + 8 * j + (lane >> 3);
            vq[2 * g + j] = (uint32_t)(min(c0 + r, N - 1) - c0) * (uint32_t)(nb * kRowBlk) +
                            (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
        }
        if constexpr (FMT == BX_TYPE_Q6_K) {
            hb[g] = weight(g) + (int64_t)N * nb * 128 + ((int64_t)c0 * nb + b0) * 64;
            const int r = 16 * u + (lane >> 2);
            vh[g] = (uint32_t)(min(c0 + r, N - 1) - c0) * (uint32_t)(nb * 64) +
                    (uint32_t)(((lane & 3) ^ ((r >> 2) & 3)) * 16);
        }
    }
    {
        const int g = FN == 2 ? lh : 0;
        const int64_t n = min(min(col0(g), N - 1) + lr, N - 1), sb = n * nb + b0;
        if constexpr (FMT == BX_TYPE_Q4_K) scp[0] = weight(g) + (int64_t)N * nb * 128 + sb * 16;
        if constexpr (FMT == BX_TYPE_Q6_K) {
            scp[0] = weight(g) + (int64_t)N * nb * 192 + sb * 16;
            scp[1] = weight(g) + (int64_t)N * nb * 208 + sb * 2;   // the dword holding it is copied
        }
        if constexpr (FMT == BX_TYPE_Q8_0) scp[0] = weight(g) + (int64_t)N * K + sb * 16;
    }

    auto issue_a = [&](int H, int slot) {
        const unsigned char* src = xb + (int64_t)min(H, nh - 1) * 256;
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lbase + slot * Sh::kSlot + wid * PA * 1024);
#pragma unroll
        for (int j = 0; j < PA; ++j) dma16(va[j], src, dst + j * 1024);
    };
    auto issue_half = [&](int H) {   // Q8_0: buffer H % NH
        if constexpr (F::kHalf > 0) {
            const int Hc = min(H, nh - 1);
            const uint32_t dst = __builtin_amdgcn_readfirstlane(rbase + (H % Sh::NH) * F::half_bytes(FN));
#pragma unroll
            for (int j = 0; j < 2 * FN; ++j)
                dma16(vq[j], qb[j >> 1] + (int64_t)Hc * 128, dst + ((j >> 1) * 4 + 2 * u + (j & 1)) * 1024);
        }
    };
    auto issue_blk = [&](int b) {    // buffer b % NB
        const int bc = min(b, nblk - 1);
        const uint32_t dst =
            __builtin_amdgcn_readfirstlane(rbase + Sh::NH * F::half_bytes(FN) + (b % Sh::NB) * F::blk_bytes(FN));
        if constexpr (F::kBlk > 0) {
#pragma unroll
            for (int j = 0; j < 2 * FN; ++j)
                dma16(vq[j], qb[j >> 1] + (int64_t)bc * 128, dst + ((j >> 1) * 4 + 2 * u + (j & 1)) * 1024);
        }
        if constexpr (FMT == BX_TYPE_Q6_K) {
#pragma unroll
            for (int j = 0; j < FN; ++j) dma16(vh[j], hb[j] + (int64_t)bc * 64, dst + R * 128 + (2 * j + u) * 1024);
            dma16p(scp[0] + bc * 16, dst + R * 192);
            dma4p(reinterpret_cast<const void*>(reinterpret_cast<uintptr_t>(scp[1] + bc * 2) & ~(uintptr_t)3),
                  dst + R * 192 + 1024);
        } else if constexpr (FMT == BX_TYPE_Q4_K) {
            dma16p(scp[0] + bc * 16, dst + R * 128);
        } else {
            dma16p(scp[0] + bc * 16, dst);
        }
    };

    f16v acc[FM][FN];
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
        for (int g = 0; g < FN; ++g)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[f][g][r] = 0.f;

    // swizzled A chunk of this lane, unit and row; chunk8 of a step XORs in
    const uint32_t abx = (uint32_t)((F::lh_chunk(lh) | F::chunk8(u, 0)) ^ (lr & 15));
    const uint32_t qx = (uint32_t)(lh ^ ((lr >> 1) & 7));
    // parity of a Q6_K scale's index among the d values (which half of its dword)
    uint32_t dpar[FN];
    if constexpr (FMT == BX_TYPE_Q6_K) {
#pragma unroll
        for (int g = 0; g < FN; ++g)
            dpar[g] = (uint32_t)((int64_t)min(min(col0(g), N - 1) + lr, N - 1) * nb + b0) & 1u;
    }

    // the loop's issue order, for the steps before 0
    static_for<-Sh::kFirst>([&](auto vc) {
        constexpr int v = Sh::kFirst + decltype(vc)::value;
        if constexpr (v + NA - 1 >= 0) issue_a(v + NA - 1, v + NA - 1);
        if constexpr (v + Sh::NH - 1 >= 0) issue_half(v + Sh::NH - 1);
        if constexpr (v % 2 == 0 && v / 2 + Sh::NB - 1 >= 0) issue_blk(v / 2 + Sh::NB - 1);
    });
    int slot = 0;
    for (int b = 0; b < nblk; ++b) {
        typename F::Scale sc[FN];
        static_for<2>([&](auto hc) {
            constexpr int h = decltype(hc)::value;
            const int H = 2 * b + h;
            wait_vm_barrier<Sh::fly(h)>();
            const int prev = slot == 0 ? NA - 1 : slot - 1;
            issue_a(H + NA - 1, prev);
            issue_half(H + Sh::NH - 1);
            if constexpr (h == 0) issue_blk(b + Sh::NB - 1);
            const unsigned char* const as = smem + slot * Sh::kSlot + lr * 256;
            const unsigned char* const rh = raw + (H % Sh::NH) * F::half_bytes(FN);
            const unsigned char* const rb = raw + Sh::NH * F::half_bytes(FN) + (b % Sh::NB) * F::blk_bytes(FN);
            if constexpr (h == 0) {
#pragma unroll
                for (int g = 0; g < FN; ++g) {
                    const int row = 32 * g + lr;
                    if constexpr (FMT == BX_TYPE_Q4_K) sc[g].h = *reinterpret_cast<const u4v*>(rb + R * 128 + row * 16);
                    if constexpr (FMT == BX_TYPE_Q8_0) sc[g].d = *reinterpret_cast<const u4v*>(rb + row * 16);
                    if constexpr (FMT == BX_TYPE_Q6_K) {
                        sc[g].sc = *reinterpret_cast<const u4v*>(rb + R * 192 + row * 16);
                        const uint32_t dd = *reinterpret_cast<const uint32_t*>(rb + R * 192 + 1024 + row * 4);
                        sc[g].d = ((dpar[g] + (uint32_t)b) & 1u) ? dd >> 16 : dd & 0xffffu;
                    }
                }
            }
            h8 bf[FN][4];
#pragma unroll
            for (int g = 0; g < FN; ++g) {
                const int row = 32 * g + lr;
                typename F::Raw r;
                if constexpr (FMT == BX_TYPE_Q4_K) {
                    r.q = *reinterpret_cast<const u4v*>(rb + row * 128 + ((uint32_t)(4 * h + 2 * u) ^ qx) * 16);
                } else if constexpr (FMT == BX_TYPE_Q6_K) {
                    r.ql = *reinterpret_cast<const u4v*>(rb + row * 128 + ((uint32_t)(4 * h + 2 * u) ^ qx) * 16);
                    r.qh = *reinterpret_cast<const u2v*>(rb + R * 128 + row * 64 +
                                                         ((2 * h + u) ^ ((lr >> 2) & 3)) * 16 + lh * 8);
                } else {
#pragma unroll
                    for (int p = 0; p < 2; ++p)
                        r.q[p] = *reinterpret_cast<const u4v*>(rh + row * 128 + ((uint32_t)(4 * u + 2 * p) ^ qx) * 16);
                }
                decode(r, sc[g], h, u, bf[g]);
            }
            // a step's A fragments are requested before the MFMAs of the step before
            h8 af[2][FM];
            auto read_a = [&](auto stc) {
                constexpr int st = decltype(stc)::value;
                const unsigned char* const ap = as + (((uint32_t)F::chunk8(0, st) ^ abx) << 4);
#pragma unroll
                for (int f = 0; f < FM; ++f) af[st & 1][f] = *reinterpret_cast<const h8*>(ap + f * 8192);
            };
            read_a(std::integral_constant<int, 0>{});
            static_for<4>([&](auto stc) {
                constexpr int st = decltype(stc)::value;
                if constexpr (st < 3) read_a(std::integral_constant<int, st + 1>{});
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int f = 0; f < FM; ++f)
#pragma unroll
                    for (int g = 0; g < FN; ++g)
                        acc[f][g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[st & 1][f], bf[g][st], acc[f][g], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            });
            slot = slot + 1 == NA ? 0 : slot + 1;
        });
    }
    // ---- the tile through LDS, FP32 rows of BN columns (group g of 128 at
    // column 128 g): the second wavefronts' sums, then the first ones' added
    wait_vm_barrier<0>();   // also the last (repeated) copies
    // D layout: lane l, register r holds row 8*(r/4) + 4*(l/32) + r%4, column l%32
    unsigned char* const sp = smem + 4 * lh * Sh::kRow + (32 * wave + lr) * 4;
    auto at = [&](int f, int g, int r) {
        return reinterpret_cast<float*>(sp + (32 * f + 8 * (r >> 2) + (r & 3)) * Sh::kRow + 512 * g);
    };
    auto each = [&](auto fn) {
#pragma unroll
        for (int f = 0; f < FM; ++f)
#pragma unroll
            for (int g = 0; g < FN; ++g)
#pragma unroll
                for (int r = 0; r < 16; ++r) fn(f, g, r);
    };
    if (u == 1) each([&](int f, int g, int r) { *at(f, g, r) = acc[f][g][r]; });
    __syncthreads();
    if (u == 0) {
        each([&](int f, int g, int r) { acc[f][g][r] += *at(f, g, r); });
        each([&](int f, int g, int r) { *at(f, g, r) = acc[f][g][r]; });
    }
    __syncthreads();
    constexpr int kQ = BN / 4;          // quads of columns per row
    constexpr int kQuads = BM * kQ;     // a multiple of kThreads
    auto quad = [&](int i) {
        return *reinterpret_cast<const f4v*>(smem + (i / kQ) * Sh::kRow + (i % kQ) * 16);
    };
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(job.part, 0, 0x7fffffff, 0x00020000);
    const int tb = (int)((int64_t)tile * S * kQuads * 16);   // the tile's partials, bytes
    if (S > 1) {
        for (int i = threadIdx.x; i < kQuads; i += kThreads)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, quad(i)), rs, tb + (s * kQuads + i) * 16, 0,
                                                   kSc1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) last = tagged_arrive(&job.cnt[tile], job.tag) == (uint32_t)S ? 1u : 0u;
        __syncthreads();
        if (!last) return;
        if (threadIdx.x == 0)
            __hip_atomic_store(&job.cnt[tile], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // the sums of the S slices, in slice order, back into the staged rows:
        // four slices of kG quads in flight per thread (a thread has 2 FM FN)
        constexpr int kPer = kQuads / kThreads, kG = kPer % 4 == 0 ? 4 : 2;
        for (int i0 = threadIdx.x; i0 < kQuads; i0 += kG * kThreads) {
            f4v sum[kG] = {};
            for (int q0 = 0; q0 < S; q0 += 4) {
                u4v v[4][kG];
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int k = 0; k < kG; ++k)
                        v[q][k] = __builtin_amdgcn_raw_buffer_load_b128(
                            rs, tb + (min(q0 + q, S - 1) * kQuads + i0 + k * kThreads) * 16, 0, kSc1);
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (q0 + q < S)
#pragma unroll
                        for (int k = 0; k < kG; ++k) sum[k] += __builtin_bit_cast(f4v, v[q][k]);
            }
#pragma unroll
            for (int k = 0; k < kG; ++k) {
                const int i = i0 + k * kThreads;
                *reinterpret_cast<f4v*>(smem + (i / kQ) * Sh::kRow + (i % kQ) * 16) = sum[k];
            }
        }
        __syncthreads();
    }

    // ---- epilogue: a thread takes four columns of a row
    const bool vec = (N & 3) == 0;   // rows start 8 (16) bytes aligned with their base
    if (two) {
        uint16_t* const Y = job.t.Y[0];
        constexpr int kH = kQ / 2;   // quads of gate columns
        for (int i = threadIdx.x; i < BM * kH; i += kThreads) {
            const int m = m0 + i / kH, n = n0 + (i % kH) * 4;
            if (m >= M || n >= N) continue;
            const unsigned char* row = smem + (i / kH) * Sh::kRow + (i % kH) * 16;
            const f4v a = *reinterpret_cast<const f4v*>(row), b = *reinterpret_cast<const f4v*>(row + kH * 16);
            uint16_t o[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float act = h2f(f2h(silu_f32(h2f(f2h(a[k])))));
                o[k] = f2h(act * h2f(f2h(b[k])));
            }
            store4(Y + (int64_t)m * N + n, o, vec, N - n);
        }
        return;
    }
    for (int i = threadIdx.x; i < kQuads; i += kThreads) {
        const int m = m0 + i / kQ, n = n0 + (i % kQ) * 4;
        if (m >= M || n >= N) continue;
        const f4v a = quad(i);
        if (epi == EPI_RESID) {
            float* const h = job.t.H + (int64_t)m * N + n;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (n + k < N) h[k] += h2f(f2h(a[k]));
        } else {
            uint16_t o[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = f2h(a[k] + (bias ? h2f(bias[min(n + k, N - 1)]) : 0.f));
            store4(job.t.Y[mem] + (int64_t)m * N + n, o, vec, N - n);
        }
    }
}

// Tile and slice plan of one launch: the least estimated time.  The model's
// constants (microseconds) are fitted to a sweep of every (FM, FN, S) over 13
// shapes of 17..2000 rows: a round of tiles costs its pipeline fill and
// epilogue plus a time per 256-element block of K (decode-bound up to FM = 2,
// then MFMA-bound), more when every CU streams; a split adds the exchange of
// its partials.  Example: 75 x 6144 x 2048 Q4_K takes 13.1 us as 32-row tiles,
// 14.7 us as 96-row tiles in 4 slices, 28 us as 96 x 256 tiles.  SwiGLU has tiles
// of 64 + 64 columns too (FN 1), for matrices whose 128 + 128 leave CUs idle: 128 x
// 3072 x 1024 Q8_0 12.5 -> 8.6 us (10.3 on the tiles of gemm.hip), 128 x 6144 x 2048
// 21.1 -> 15.7.
//
// The slices decide the order in which an output's sums are added.  A residual
// launch has those of the plain launch, being planned alike, and SwiGLU takes
// those of the plain launch of gate or up: both give the bits of the separate
// ops.  q / k / v in one launch have slices of their own: those of the separate
// launches, which fill the chip three times over, cost up to twice the time (200
// rows of 2048 + 1024 + 1024 columns, K = 2048, Q4_K 12.9 us against 28.8), so a
// group's sums may differ from the plain launches' in the last bits of FP32.
struct QPlan {
    int fm, fn, S;
};

QPlan quant_plan(const TileJob& job, int wtype, int epi, int M, int K, bool have_ws) {
    static constexpr double kFill[2][4] = {{1.3, 3.4, 3.8, 4.4}, {1.5, 5.0, 7.0, 8.0}};
    static constexpr double kBlock[2][4] = {{1.17, 1.17, 1.5, 1.78}, {2.1, 2.15, 2.4, 2.9}};
    const int cus = num_cus(), nb = K / 256;
    const bool two = epi == EPI_SWIGLU;
    int from = 1, to = have_ws ? std::min(16, nb) : 1;
    if (two && have_ws) from = to = quant_plan(job, wtype, EPI_STORE, M, K, have_ws).S;
    QPlan best{1, 1, from};
    double least = 1e30;
    for (int fn = 1; fn <= 2; ++fn) {
        // 96 rows at most with Q6_K at 256 columns: its raw blocks take the LDS
        const int fm_max = wtype == BX_TYPE_Q6_K && fn == 2 ? 3 : 4;
        for (int fm = 1; fm <= fm_max; ++fm) {
            int64_t tiles = 0;
            const int bn = two ? 64 * fn : 128 * fn;
            for (int i = 0; i < job.members; ++i) tiles += (job.N[i] + bn - 1) / bn;
            tiles *= (M + 32 * fm - 1) / (32 * fm);
            for (int S = from; S <= to; ++S) {
                // more slices than fill the CUs only where they are given.  The
                // partials then fit as 32-row tiles at the latest: of the plain
                // launch, at most cus tiles of 128 x 256, SwiGLU's are twice
                if (S > 1 && ((tiles * S > cus && from < to) || tiles > kSplGroups ||
                              tiles * S * fm * fn * 4096 > kSplFloats))
                    break;
                const int64_t wgs = tiles * S;
                double block = kBlock[fn - 1][fm - 1] * (wtype == BX_TYPE_Q6_K ? 1.35 : 1.0);
                if (wgs > cus * 7 / 8) block *= 1.0 + 0.06 * fm * fn;
                const double rounds = wgs <= cus ? 1.0 : (double)((wgs + cus - 1) / cus);
                double t = rounds * (kFill[fn - 1][fm - 1] + (nb + S - 1) / S * block) +
                                 (S > 1 ? 2.0 + 0.9 * fm * fn + 0.3 * S : 0.0);
                if (two && fn == 1) t *= 1.05;   // a tie goes to the tiles that read X half as often
                if (t < least) {
                    least = t;
                    best = QPlan{fm, fn, S};
                }
            }
        }
    }
    return best;
}

template <int FMT, int FM, int FN>
int launch_quant(QuantJob job, const uint16_t* bias, const uint16_t* X, int M, int K, int epi, hipStream_t st) {
    using Sh = QShape<FMT, FM, FN>;
    const int cn = epi == EPI_SWIGLU ? Sh::BN / 2 : Sh::BN;
    job.t.tiles_m = (M + Sh::BM - 1) / Sh::BM;
    int64_t tiles = 0;
    for (int i = 0; i < job.t.members; ++i) {
        job.t.tiles_n[i] = (job.t.N[i] + cn - 1) / cn;
        tiles += job.t.tiles_n[i];
    }
    tiles *= (int64_t)job.t.tiles_m * job.S;
    if (tiles > (1 << 30)) return fail(BX_EINVAL, "gemm: too many tiles");
    const void* fn = reinterpret_cast<const void*>(&gemm_quant_kernel<FMT, FM, FN>);
    static std::atomic<uint64_t> allowed{0};
    if (int rc = allow_lds(allowed, fn, Sh::kLds, "gemm quant: LDS attribute")) return rc;
    gemm_quant_kernel<FMT, FM, FN><<<dim3((unsigned)tiles), kThreads, Sh::kLds, st>>>(job, X, bias, M, K, epi);
    return launch_check("gemm_quant");
}

template <int FMT>
int quant_typed(const QPlan& p, const QuantJob& job, const uint16_t* bias, const uint16_t* X, int M, int K, int epi,
                hipStream_t st) {
    if (p.fn == 1) {
        switch (p.fm) {
            case 1: return launch_quant<FMT, 1, 1>(job, bias, X, M, K, epi, st);
            case 2: return launch_quant<FMT, 2, 1>(job, bias, X, M, K, epi, st);
            case 3: return launch_quant<FMT, 3, 1>(job, bias, X, M, K, epi, st);
            default: return launch_quant<FMT, 4, 1>(job, bias, X, M, K, epi, st);
        }
    }
    switch (p.fm) {
        case 1: return launch_quant<FMT, 1, 2>(job, bias, X, M, K, epi, st);
        case 2: return launch_quant<FMT, 2, 2>(job, bias, X, M, K, epi, st);
        case 3: return launch_quant<FMT, 3, 2>(job, bias, X, M, K, epi, st);
        default:
            if constexpr (FMT != BX_TYPE_Q6_K) return launch_quant<FMT, 4, 2>(job, bias, X, M, K, epi, st);
            else return launch_quant<FMT, 3, 2>(job, bias, X, M, K, epi, st);
    }
}

}  // namespace

// Whether the kernel takes a launch: K in whole 256-element blocks, operands
// aligned for 16-byte copies; Q6_K scales are copied as aligned dwords of two,
// so their count must be even.
bool gemm_quant_ok(int wtype, const TileJob& job, const uint16_t* X, int M, int K) {
    if (M <= 16 || K % 256 != 0 || (reinterpret_cast<uintptr_t>(X) & 15)) return false;
    if (wtype != BX_TYPE_Q4_K && wtype != BX_TYPE_Q6_K && wtype != BX_TYPE_Q8_0) return false;
    for (int i = 0; i < 3; ++i)
        if (reinterpret_cast<uintptr_t>(job.W[i]) & 15) return false;   // absent ones are null
    for (int i = 0; i < job.members; ++i)
        if (wtype == BX_TYPE_Q6_K && ((int64_t)job.N[i] * (K / 256)) % 2 != 0) return false;
    return true;
}

// {rows, columns, K slices} of a launch's tiles
void gemm_quant_shape(int wtype, int epi, const TileJob& job, int M, int K, bool have_ws, int* shape) {
    const QPlan p = quant_plan(job, wtype, epi, M, K, have_ws);
    shape[0] = 32 * p.fm;
    shape[1] = 128 * p.fn;
    shape[2] = p.S;
}

int gemm_quant(int wtype, int epi, const TileJob& t, const uint16_t* bias, const uint16_t* X, int M, int K, void* ws,
               size_t wsb, hipStream_t st) {
    const bool have_ws = ws != nullptr && wsb >= kSplCntBytes + (size_t)kSplFloats * 4;
    const QPlan p = quant_plan(t, wtype, epi, M, K, have_ws);
    QuantJob job{};
    job.t = t;
    job.S = p.S;
    if (p.S > 1) {
        job.cnt = static_cast<uint64_t*>(ws);
        job.part = reinterpret_cast<float*>(static_cast<unsigned char*>(ws) + kSplCntBytes);
        job.tag = next_launch_tag();
    }
    switch (wtype) {
        case BX_TYPE_Q4_K: return quant_typed<BX_TYPE_Q4_K>(p, job, bias, X, M, K, epi, st);
        case BX_TYPE_Q6_K: return quant_typed<BX_TYPE_Q6_K>(p, job, bias, X, M, K, epi, st);
        case BX_TYPE_Q8_0: return quant_typed<BX_TYPE_Q8_0>(p, job, bias, X, M, K, epi, st);
        default: return fail(BX_EUNSUPPORTED, "gemm: unsupported type");
    }
}

}  // namespace bx
