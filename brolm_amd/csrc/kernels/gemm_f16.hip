// Linear on FP16 weights for 17 rows and more, on MFMA (v_mfma_f32_32x32x16_f16):
// Y[M,N] = X[M,K] W[N,K]^T, K a multiple of 64.
//
// A workgroup of WM x WN wavefronts computes a BM x BN tile, each wavefront a
// (BM / WM) x 64 part as 32x32 fragments.  K advances 64 per stage through NB
// LDS buffers filled by LDS-DMA (no registers between HBM and LDS), whole
// 128-byte lines of a row at a time, 16-byte chunks XOR-swizzled by the row.
// A stage is four steps of 16; a step's fragments are requested while the step
// before multiplies, in an order fixed with scheduling barriers (left to the
// compiler, every read was waited for right after its issue).  One barrier a
// stage, before the last step: by then every wavefront has read the buffer,
// so the copies of the stage NB ahead go into it, and the next stage's first
// fragments are read under the last step's MFMAs.
//
// What bounds it: the matrix cores, busy for 73 % of the cycles at 256 x 256 tiles
// (SwiGLU 2048 x 12288 x 4096), at a clock that falls to 1.6 GHz under this load;
// the LDS is active for 29 % (192 KB of fragments a stage), a third of the wave
// cycles wait.  128 x 128 tiles read 1.5 times as much LDS for the same MFMAs, but
// fill the chip where 256 x 256 does not; the launcher estimates the time of each
// shape.
//
// The epilogue stages the FP16 tile in LDS and stores 16 bytes a thread, rows
// of whole lines; at any alignment, so odd column counts take the same stores
// (one by one they made SwiGLU 700 x 1500 x 768 16.1 us, 10.9 with them).
#include <algorithm>

#include "gemm_job.h"

namespace bx {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef u4v __attribute__((aligned(2))) any16;   // eight FP16 values at any address
typedef float f4v __attribute__((ext_vector_type(4)));
typedef f4v __attribute__((aligned(4))) any_f4;

template <int BM_, int WM_, int WN_, int NB_>
struct FShape {
    static constexpr int BM = BM_, WM = WM_, WN = WN_, NB = NB_;
    static constexpr int BN = 64 * WN, NW = WM * WN, NT = 64 * NW;
    static constexpr int FM = BM / WM / 32, FN = 2;
    static constexpr int PA = BM / 8 / NW, PB = BN / 8 / NW, P = PA + PB;   // copies per wavefront and stage
    static constexpr int kStage = (BM + BN) * 128;
    static constexpr int kRow = BN * 2 + 16;   // epilogue: bytes of a staged FP16 row
    static constexpr int kLds = NB * kStage > BM * kRow ? NB * kStage : BM * kRow;
    static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0 && kLds <= 160 * 1024);
};

template <class Sh>
__global__ __launch_bounds__(Sh::NT, 1) void gemm_f16_kernel(TileJob job, const uint16_t* __restrict__ X,
                                                            const uint16_t* __restrict__ bias, int M, int K, int epi) {
    constexpr int BM = Sh::BM, BN = Sh::BN, FM = Sh::FM, FN = Sh::FN, NB = Sh::NB, PA = Sh::PA, PB = Sh::PB, P = Sh::P;
    extern __shared__ __align__(1024) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int tiles = 0;
    for (int i = 0; i < job.members; ++i) tiles += job.tiles_n[i];
    const int t = xcd_tile((int)blockIdx.x, job.tiles_m * tiles);
    int tn = t / job.tiles_m, mem = 0;
    while (tn >= job.tiles_n[mem]) tn -= job.tiles_n[mem++];
    const bool two = epi == EPI_SWIGLU;   // fragment column g of a wavefront: gate, up
    const int N = job.N[mem];
    const int m0 = (t % job.tiles_m) * BM, n0 = tn * (two ? BN / 2 : BN);

    // ---- sources of the copies: eight rows of 128 bytes each.  Rows past M
    // or N repeat the last one (their results are not stored).  Row r of the W
    // part: column 64 w + 32 g + i of the tile is wavefront column w's fragment g
    const uint32_t lbase = lds_addr(smem);
    const int drow = lane >> 3;
    uint32_t va[PA], vb[PB];
    const unsigned char* const xb = reinterpret_cast<const unsigned char*>(X + (int64_t)m0 * K);
    const unsigned char* wb[PB];
#pragma unroll
    for (int j = 0; j < PA; ++j) {
        const int r = 8 * (wave * PA + j) + drow;
        va[j] = (uint32_t)(min(m0 + r, M - 1) - m0) * (uint32_t)K * 2u + (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
    }
#pragma unroll
    for (int j = 0; j < PB; ++j) {
        const int r0 = 8 * (wave * PB + j), r = r0 + drow;
        const int g = (r0 >> 5) & 1;   // wave-uniform
        const int c = two ? 32 * (r >> 6) + (r & 31) : r;
        wb[j] = static_cast<const unsigned char*>(two ? job.W[g] : job.W[mem]) + (int64_t)n0 * K * 2;
        vb[j] = (uint32_t)(min(n0 + c, N - 1) - n0) * (uint32_t)K * 2u + (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
    }
    const int nk = K / 64;
    auto issue1 = [&](int64_t ko, uint32_t dst, auto jc) {
        constexpr int j = decltype(jc)::value;
        if constexpr (j < PA) dma16(va[j], xb + ko, dst + (wave * PA + j) * 1024);
        else dma16(vb[j - PA], wb[j - PA] + ko, dst + BM * 128 + (wave * PB + j - PA) * 1024);
    };
    auto stage_at = [&](int buf) { return (uint32_t)__builtin_amdgcn_readfirstlane(lbase + buf * Sh::kStage); };
    auto k_off = [&](int kt) { return (int64_t)min(kt, nk - 1) * 128; };

    // ---- fragments: lane l holds row l % 32, k [8 (l / 32), + 8) of a step
    const int lr = lane & 31, lh = lane >> 5, sw = (lr >> 1) & 7;
    const int ao = ((wave / Sh::WN) * 32 * FM + lr) * 128, bo = BM * 128 + ((wave % Sh::WN) * 64 + lr) * 128;
    const int cs[4] = {(lh ^ sw) * 16, ((2 + lh) ^ sw) * 16, ((4 + lh) ^ sw) * 16, ((6 + lh) ^ sw) * 16};
    f16v acc[FM][FN];
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
        for (int g = 0; g < FN; ++g)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[f][g][r] = 0.f;
    struct Frags {
        h8 a[FM], b[FN];
    };
    constexpr int NM = FM * FN, NR = FM + FN;
    auto read1 = [&](Frags& x, const unsigned char* p, auto ic) {
        constexpr int i = decltype(ic)::value;
        if constexpr (i < FN) x.b[i] = *reinterpret_cast<const h8*>(p + bo + i * 4096);
        else x.a[i - FN] = *reinterpret_cast<const h8*>(p + ao + (i - FN) * 4096);
    };
    // one step: MFMA i of the step's fragments `use`, then the reads of the
    // next step's and whatever else falls to slot i.  W is the first operand, so
    // a lane's results are four consecutive columns of one row (D layout: rows
    // 8 (r / 4) + 4 (l / 32) + r % 4 are columns of Y, column l % 32 its row).
    auto step = [&](const Frags& use, Frags& next, const unsigned char* p, auto extra) {
        static_for<NM>([&](auto ic) {
            constexpr int i = decltype(ic)::value, f = i / FN, g = i % FN;
            acc[f][g] = __builtin_amdgcn_mfma_f32_32x32x16_f16(use.b[g], use.a[f], acc[f][g], 0, 0, 0);
            static_for<NR>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                if constexpr (r * (NM > 2 ? NM - 2 : 1) / NR == i) read1(next, p, rc);
            });
            extra(ic);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto none = [](auto) {};

    static_for<NB - 1>([&](auto bc) {
        constexpr int b = decltype(bc)::value;
        static_for<P>([&](auto jc) { issue1(k_off(b), stage_at(b), jc); });
    });
    wait_vm_barrier<P*(NB - 2)>();
    static_for<P>([&](auto jc) { issue1(k_off(NB - 1), stage_at(NB - 1), jc); });
    Frags x, y;
    static_for<NR>([&](auto ic) { read1(x, smem + cs[0], ic); });
    int cur = 0;
    for (int kt = 0; kt < nk; ++kt) {
        const unsigned char* const p = smem + cur * Sh::kStage;
        const int nx = cur + 1 == NB ? 0 : cur + 1;
        step(x, y, p + cs[1], none);
        step(y, x, p + cs[2], none);
        step(x, y, p + cs[3], none);
        wait_vm_barrier<P*(NB - 2)>();
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t dst = stage_at(cur);
        const int64_t ko = k_off(kt + NB);
        step(y, x, smem + nx * Sh::kStage + cs[0], [&](auto ic) {
            static_for<P>([&](auto jc) {
                if constexpr (decltype(jc)::value * NM / P == decltype(ic)::value) issue1(ko, dst, jc);
            });
        });
        cur = nx;
    }

    // ---- epilogue: the FP16 tile in LDS (gate columns, then up columns), then rows
    wait_vm_barrier<0>();   // the last (repeated) copies too
    const int wn = wave % Sh::WN;
    auto col = [&](int g) { return two ? (BN / 2) * g + 32 * wn : 64 * wn + 32 * g; };
    const bool add_bias = epi == EPI_STORE && bias != nullptr;
#pragma unroll
    for (int g = 0; g < FN; ++g) {
        const int c = col(g) + 4 * lh;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float bv[4] = {0.f, 0.f, 0.f, 0.f};
            if (add_bias)
#pragma unroll
                for (int k = 0; k < 4; ++k) bv[k] = h2f(bias[min(n0 + c + 8 * q + k, N - 1)]);
#pragma unroll
            for (int f = 0; f < FM; ++f) {
                const f16v& a = acc[f][g];
                const u2v w = {(uint32_t)f2h(a[4 * q] + bv[0]) | ((uint32_t)f2h(a[4 * q + 1] + bv[1]) << 16),
                               (uint32_t)f2h(a[4 * q + 2] + bv[2]) | ((uint32_t)f2h(a[4 * q + 3] + bv[3]) << 16)};
                *reinterpret_cast<u2v*>(smem + ((wave / Sh::WN) * 32 * FM + 32 * f + lr) * Sh::kRow + (c + 8 * q) * 2) = w;
            }
        }
    }
    __syncthreads();
    constexpr int kChunks = BN / 8;
    const int cn = two ? kChunks / 2 : kChunks;   // chunks of output columns
    uint16_t* const Y = two ? job.Y[0] : job.Y[mem];
    for (int i = threadIdx.x; i < BM * cn; i += Sh::NT) {
        const int row = i / cn, m = m0 + row, n = n0 + (i % cn) * 8;
        if (m >= M || n >= N) continue;
        const unsigned char* const src = smem + row * Sh::kRow + (i % cn) * 16;
        union {
            u4v v;
            uint16_t h[8];
        } o;
        o.v = *reinterpret_cast<const u4v*>(src);
        if (two) {
            union {
                u4v v;
                uint16_t h[8];
            } up;
            up.v = *reinterpret_cast<const u4v*>(src + BN);
#pragma unroll
            for (int k = 0; k < 8; ++k) o.h[k] = f2h(h2f(f2h(silu_f32(h2f(o.h[k])))) * h2f(up.h[k]));
        }
        const int64_t at = (int64_t)m * N + n;
        if (epi == EPI_RESID) {
            float* const h = job.H + at;
            if (n + 8 <= N) {
                f4v a = *reinterpret_cast<any_f4*>(h), b = *reinterpret_cast<any_f4*>(h + 4);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    a[k] += h2f(o.h[k]);
                    b[k] += h2f(o.h[4 + k]);
                }
                *reinterpret_cast<any_f4*>(h) = a;
                *reinterpret_cast<any_f4*>(h + 4) = b;
            } else {
#pragma unroll
                for (int k = 0; k < 7; ++k)
                    if (n + k < N) h[k] += h2f(o.h[k]);
            }
        } else if (n + 8 <= N) {
            *reinterpret_cast<any16*>(Y + at) = o.v;
        } else {
#pragma unroll
            for (int k = 0; k < 7; ++k)
                if (n + k < N) Y[at + k] = o.h[k];
        }
    }
}

template <class Sh>
int launch(TileJob job, const uint16_t* bias, const uint16_t* X, int M, int K, int epi, hipStream_t st) {
    const int cn = epi == EPI_SWIGLU ? Sh::BN / 2 : Sh::BN;
    job.tiles_m = (M + Sh::BM - 1) / Sh::BM;
    int64_t tiles = 0;
    for (int i = 0; i < job.members; ++i) {
        job.tiles_n[i] = (job.N[i] + cn - 1) / cn;
        tiles += job.tiles_n[i];
    }
    tiles *= job.tiles_m;
    if (tiles > (1 << 30)) return fail(BX_EINVAL, "gemm: too many tiles");
    const void* fn = reinterpret_cast<const void*>(&gemm_f16_kernel<Sh>);
    static std::atomic<uint64_t> allowed{0};
    if (int rc = allow_lds(allowed, fn, Sh::kLds, "gemm f16: LDS attribute")) return rc;
    gemm_f16_kernel<Sh><<<dim3((unsigned)tiles), Sh::NT, Sh::kLds, st>>>(job, X, bias, M, K, epi);
    return launch_check("gemm_f16");
}

using T256 = FShape<256, 2, 4, 2>;   // 256 x 256, 8 wavefronts
using T128 = FShape<256, 4, 2, 3>;   // 256 x 128, 8 wavefronts
using S128 = FShape<128, 2, 2, 4>;   // 128 x 128, 4 wavefronts, one workgroup per CU
using S128x2 = FShape<128, 2, 2, 2>; // the same with two buffers, two workgroups per CU
using S64 = FShape<128, 4, 1, 4>;    // 128 x 64, 4 wavefronts
using Q64 = FShape<64, 2, 1, 6>;     // 64 x 64, 2 wavefronts

}  // namespace

int gemm_f16_small(int epi, const TileJob& job, const uint16_t* bias, const uint16_t* X, int M, int K, hipStream_t st);

// K in whole stages, operands aligned for 16-byte copies.
bool gemm_f16_ok(const TileJob& job, const uint16_t* X, int M, int K) {
    if (M <= 16 || K % 64 != 0 || (reinterpret_cast<uintptr_t>(X) & 15)) return false;
    for (int i = 0; i < 3; ++i)
        if (reinterpret_cast<uintptr_t>(job.W[i]) & 15) return false;   // absent ones are null
    return true;
}

// The tile shape with the least estimated time: rounds of tiles over the chip,
// each a fill (with the epilogue) and a time per stage that grows with the
// share of the CUs at work (LDS and L2 contention, and the clock, which falls
// from 2.4 to 1.6 GHz under full MFMA load).  Constants in microseconds,
// fitted to 19 shapes of 30..2048 rows.  Some of them (TFLOP/s by shape, with
// the register-staged tiles that ran before in brackets): SwiGLU 2048 x 12288
// x 4096: 256 x 256 1116, 256 x 128 1033, 128 x 128 1001 [815]; 2000 x 4096 x
// 2048: 256 x 128 856, 256 x 256 699 [744]; 2000 x 2048 x 6144: 128 x 128 869,
// 256 x 128 718 [649]; 777 x 2048 x 6144: 128 x 64 560, 128 x 128 444 [379].
//
// From 128 rows on and K up to 1024, up to two 64 x 64 tiles a CU also have the
// register-staged tiles of gemm.hip, four wavefronts each (the same bits: one
// 32x32x16 MFMA order over K): a shorter fill and epilogue, slower stages.  In us,
// those against the best shape here: 200 x 1000 x 768 6.9 / 7.8, 300 x 2048 x 1024
// 8.4 / 8.9, SwiGLU 300 x 3072 x 1024 11.2 / 12.8; 200 x 1024 x 2048 12.8 / 12.6, 511
// x 512 x 4096 35.0 / 20.4.
namespace {

struct Plan {
    int bm, bn, per_cu;
    double fill, idle, full;   // us a stage with few CUs at work, with all
    int (*run)(TileJob, const uint16_t*, const uint16_t*, int, int, int, hipStream_t);
};

// Null: the tiles of gemm.hip.
const Plan* f16_plan(int epi, const TileJob& job, int M, int K) {
    static const Plan kPlans[] = {
        {256, 256, 1, 12.0, 1.00, 1.65, launch<T256>}, {256, 128, 1, 9.0, 0.58, 0.92, launch<T128>},
        {128, 128, 1, 7.5, 0.37, 0.51, launch<S128>},  {128, 128, 2, 8.0, 0.57, 0.97, launch<S128x2>},
        {128, 64, 1, 5.5, 0.28, 0.31, launch<S64>},    {64, 64, 1, 4.5, 0.25, 0.27, launch<Q64>},
    };
    const Plan* best = nullptr;
    double least = 1e30;
    for (const Plan& p : kPlans) {
        const int cn = epi == EPI_SWIGLU ? p.bn / 2 : p.bn;
        int64_t tiles = 0;
        for (int i = 0; i < job.members; ++i) tiles += (job.N[i] + cn - 1) / cn;
        tiles *= (M + p.bm - 1) / p.bm;
        const int64_t slots = (int64_t)num_cus() * p.per_cu, rounds = tiles / slots, rest = tiles % slots;
        const double nk = K / 64;
        const double t = rounds * (p.fill + nk * p.full) +
                         (rest ? p.fill + nk * (p.idle + (p.full - p.idle) * (double)rest / (double)slots) : 0.0);
        if (t < least) {
            least = t;
            best = &p;
        }
    }
    if (M >= 128 && K <= 1024) {
        const int cn = epi == EPI_SWIGLU ? 32 : 64;
        int64_t tiles = 0;
        for (int i = 0; i < job.members; ++i) tiles += (job.N[i] + cn - 1) / cn;
        tiles *= (M + 63) / 64;
        if (tiles <= 2 * (int64_t)num_cus()) {
            const double t = 3.4 + (K / 64) * (tiles <= num_cus() ? 0.305 : 0.47);
            if (t < least) return nullptr;
        }
    }
    return best;
}

}  // namespace

int gemm_f16_tiles(int epi, const TileJob& job, const uint16_t* bias, const uint16_t* X, int M, int K, hipStream_t st) {
    const Plan* p = f16_plan(epi, job, M, K);
    return p ? p->run(job, bias, X, M, K, epi, st) : gemm_f16_small(epi, job, bias, X, M, K, st);
}

// {rows, columns, workgroups per CU} of a launch's tiles; false: those of gemm.hip
bool gemm_f16_shape(int epi, const TileJob& job, int M, int K, int* shape) {
    const Plan* p = f16_plan(epi, job, M, K);
    if (p) shape[0] = p->bm, shape[1] = p->bn, shape[2] = p->per_cu;
    return p != nullptr;
}

}  // namespace bx
