// Prefill / encode attention on the matrix cores (flash attention), for
// L >= 16 query rows: the L > 1 form of brotensor flash_attention_decode
// (reference src/detail/dense_decoder.cpp:606-607, causal with the query rows
// at positions valid_len - L ...) and flash_attention_gqa_forward
// (dense_decoder.cpp:737-745, causal or bidirectional).
//
// A workgroup of four wavefronts works on one KV head.  A wavefront holds 32
// query rows of one head in registers; 4 / KS wavefronts take different rows
// and heads of the group (they share every key tile), KS wavefronts the same
// rows over different keys of a tile, merged at the end (small problems, where
// the serial walk over the keys is what takes the time).  Keys and values come
// in tiles by LDS-DMA, double buffered, rows as stored, 16-byte chunks
// XOR-swizzled by the key.  Per step of NK fragments of 32 keys (two where a
// wavefront has all 64 of a tile, else one), on v_mfma_f32_32x32x16_f16:
//   S^T = K Q^T     (a lane holds 16 of a fragment's 32 keys of its query)
//   online softmax  (base-2 exponent, running max per query in FP32, moved only
//                    when some step's max exceeds it by more than 2^8; a lane
//                    sums its own keys, the halves of a query add at the end).
//                    The max of 64 keys and not of 32: the weight of the
//                    largest key so far is exactly 1 in FP16 more often, which
//                    is 0.8 % of the error of 2048 causal rows
//   O^T += V^T P^T  (P to FP16 in registers: the S^T layout is the B operand's
//                    with the keys of a k-slot group in a fixed order; V^T
//                    comes out of the row-major tile by transposing LDS reads,
//                    four keys of a column each, in that order)
//
// What bounds it: per 32 keys of a wavefront about 512 cycles of MFMA and 450
// of softmax arithmetic (half of them the exponentials, at quarter rate),
// overlapped in part by the two wavefronts of each SIMD (two workgroups per CU):
// 2048 causal rows keep VALU busy for 44 % and the matrix cores for 38 % of the
// cycles, the LDS for 19 % (one fragment of K feeds 32 queries).  Few rows (KS 4)
// have one wavefront a SIMD and wait: VALU 23 %, MFMA 9 %.  Measured against 16-row fragments with tiles staged
// through registers and V transposed on its way into LDS: 2048 causal rows of
// 32 / 8 heads of 128 100 -> 51.7 us (660 TFLOP/s), 500 rows bidirectional
// of 16 heads 17.8 -> 9.3 us, 700 rows after 2000 of 16 heads 87 -> 36 us,
// 64 rows after 2000 of 16 heads 62 -> 12.1 us.  Up to 128 keys are one tile and
// have a kernel of their own (fa_one_tile_kernel): a fragment of 32 rows has
// twice the serial work of one of 16, and a merge costs 0.5 to 0.9 us.
#include <algorithm>

#include "attention_core.h"
#include "gemm_job.h"

namespace bx {
namespace {

typedef _Float16 fa_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 fa_h4 __attribute__((ext_vector_type(4)));
typedef short fa_s4 __attribute__((ext_vector_type(4)));
typedef float fa_f16 __attribute__((ext_vector_type(16)));
typedef float fa_f4 __attribute__((ext_vector_type(4)));

constexpr int kFaThreads = 256;

template <int HD, int KS, int NK>
struct FaShape {
    static constexpr int TK = KS == 4 ? 128 : 64;       // keys per tile
    static constexpr int WK = TK / KS;                  // keys per wavefront and tile
    static_assert(WK == 32 * NK);                       // NK fragments of 32 keys
    static constexpr int RB = HD * 2;                   // bytes per key row
    static constexpr int CH = HD / 8;                   // 16-byte chunks per key row
    static constexpr int RPC = 1024 / RB;               // rows per copy instruction
    static constexpr int P = TK / RPC / 4;              // copies per wavefront and tile, of K and of V
    static constexpr int kTile = TK * RB;               // bytes of a K (or V) tile
    static constexpr int kBuf = 2 * kTile;
    static constexpr int QW = HD / 8 / KS;              // quads of O^T a wavefront finishes
    static constexpr int kRec = (HD / 8 - QW + 1) * 64; // 16-byte words of a wavefront's end-merge record
    static constexpr int kMerge = KS > 1 ? 4 * kRec * 16 : 0;
    static constexpr int kLds = 2 * kBuf > kMerge ? 2 * kBuf : kMerge;
    // chunk c of key k sits at c ^ swz(k): the 16 keys a K read covers land on
    // distinct chunks of the banks, and so do the 4 keys of a transposing read
    static __device__ __forceinline__ int swz(int k) {
        return CH == 16 ? ((k & 3) << 2) | ((k >> 2) & 3) : (k >> 1) & 7;
    }
};

// Eight and four halves at any 2-byte address (one global access of 16 and 8
// bytes: the target's unaligned access mode).
typedef u4v __attribute__((aligned(2))) fa_any16;
typedef u2v __attribute__((aligned(2))) fa_any8;

// The larger of a query's two lanes (l and l ^ 32), in both.
__device__ __forceinline__ float fa_pair_max(float v) { return fmaxf(v, __shfl_xor(v, 32)); }

// AL: K and V are 16-byte aligned.  LDS-DMA takes no others; their tiles go
// through registers, loaded before a tile's arithmetic and stored after it
// (2048 rows of 32 / 8 heads of 128, every key visible: 77 us aligned, 90 on 8
// bytes, 106 on 2; in 2-byte loads waited for at once 203 and 228).  KS = 4 holds one workgroup a
// CU by its LDS, so its 64 registers in flight have room.
template <int HD, int KS, int NK, bool AL>
__global__ __launch_bounds__(kFaThreads, !AL && KS == 4 ? 1 : 2) void fa_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ Kc,
                                                          const uint16_t* __restrict__ Vc, int L, int valid_len,
                                                          int n_q, int n_kv, int bidir, int gb, int mirror, int nsp,
                                                          float* __restrict__ recs, uint16_t* __restrict__ out) {
    using S = FaShape<HD, KS, NK>;
    constexpr int ND = HD / 32;
    extern __shared__ __align__(1024) unsigned char smem[];

    // block -> (row tile, head set): latest rows first (they see the most
    // keys); blocks from `mirror` on, the second of each CU where the grid
    // just fits two per CU, take the remaining row tiles from the lightest up
    const int G = n_q / n_kv, splits = G / gb, ny = n_kv * splits;
    // (sp > 1: sp blocks in turn share a row tile's key tiles)
    const int sp = KS == 4 ? nsp : 1;
    int b = (int)blockIdx.x / sp;
    const int part = (int)blockIdx.x % sp;
    if (b >= mirror) b = mirror + (int)gridDim.x - 1 - b;
    const int rg = 4 / KS / gb, BR = 32 * rg;     // row groups and rows per workgroup
    const int rt = (L + BR - 1) / BR - 1 - b / ny, y = b % ny;
    const int g = y / splits;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int qw = wave / KS, kw = wave % KS;     // (rows, head) of the wavefront, its keys of a tile
    const int head = g * G + (y % splits) * gb + qw % gb;
    const int lq = lane & 31, lh = lane >> 5;
    const int p0 = valid_len - L;  // position of query row 0
    const int64_t qstride = (int64_t)n_q * HD, kvstride = (int64_t)n_kv * HD;
    const int row0 = rt * BR + 32 * (qw / gb), row = row0 + lq;
    const int kend = bidir ? valid_len : min(valid_len, p0 + rt * BR + BR);
    const int nkb = (kend + S::TK - 1) / S::TK;
    const int last_key = bidir ? valid_len - 1 : min(p0 + row, valid_len - 1);
    // keys every query of the wavefront sees (its first row's)
    const int all_see = bidir ? valid_len - 1 : min(p0 + row0, valid_len - 1);
    // keys some query of the wavefront sees; none where its rows end above it
    const int any_see = bidir ? valid_len - 1 : min(p0 + row0 + 31, valid_len - 1);

    // ---- copies: wavefront w takes rows RPC (w P + j) .. of a tile
    const uint32_t lbase = lds_addr(smem);
    const unsigned char* const kb0 = reinterpret_cast<const unsigned char*>(Kc + (int64_t)g * HD);
    const unsigned char* const vb0 = reinterpret_cast<const unsigned char*>(Vc + (int64_t)g * HD);
    const int drow = lane / S::CH, dch = lane % S::CH;
    u4v kreg[AL ? 1 : S::P], vreg[AL ? 1 : S::P];   // the next tile, on its way to LDS
    auto issue = [&](int kb, int buf) {
        const int k0 = kb * S::TK, left = valid_len - 1 - k0;   // keys past the end repeat the last one
        const int64_t base = (int64_t)k0 * kvstride * 2;
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lbase + buf * S::kBuf + wave * S::P * 1024);
#pragma unroll
        for (int j = 0; j < S::P; ++j) {
            const int r = S::RPC * (wave * S::P + j) + drow;
            const uint32_t off = (uint32_t)min(r, left) * (uint32_t)(kvstride * 2) + (uint32_t)((dch ^ S::swz(r)) * 16);
            if constexpr (AL) {
                dma16(off, kb0 + base, dst + j * 1024);
                dma16(off, vb0 + base, dst + S::kTile + j * 1024);
            } else {
                kreg[j] = *reinterpret_cast<const fa_any16*>(kb0 + base + off);
                vreg[j] = *reinterpret_cast<const fa_any16*>(vb0 + base + off);
            }
        }
    };
    auto land = [&](int buf) {   // the tile issued last, where no copy brings it
        if constexpr (!AL) {
#pragma unroll
            for (int j = 0; j < S::P; ++j) {
                unsigned char* const d = smem + buf * S::kBuf + (wave * S::P + j) * 1024 + lane * 16;
                *reinterpret_cast<u4v*>(d) = kreg[j];
                *reinterpret_cast<u4v*>(d + S::kTile) = vreg[j];
            }
        }
    };

    auto tile_wait = [] {   // this tile's readers are done and the next one is there
        if constexpr (AL)
            wait_vm_barrier<0>();
        else
            __syncthreads();
    };

    // the query rows: B operand, lane l holds query l % 32, d 16 s + 8 (l / 32) ..
    fa_h8 qf[HD / 16];
    {
        const uint16_t* qrow = q + (int64_t)min(row, L - 1) * qstride + (int64_t)head * HD + 8 * lh;
#pragma unroll
        for (int s = 0; s < HD / 16; ++s)
            qf[s] = __builtin_bit_cast(fa_h8, (u4v)*reinterpret_cast<const fa_any16*>(qrow + 16 * s));
        // waited for here: left to their first use, inside the loop, the wait
        // would also cover the tile copies just issued there, every iteration
#pragma unroll
        for (int s = 0; s < HD / 16; ++s) asm volatile("" : "+v"(qf[s]));
    }
    fa_f16 o[ND];   // O^T: d = 32 j + 8 (r / 4) + 4 lh + r % 4 of query lq
#pragma unroll
    for (int j = 0; j < ND; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[j][r] = 0.f;
    float m = -INFINITY, l = 0.f;   // running max (base-2 units), sum over this lane's keys
    const float sl2 = 1.4426950408889634f / sqrtf((float)HD);

    // LDS addresses: K rows of 32 keys (A operand: lane l holds key l % 32,
    // d 16 s + 8 (l / 32)); transposing reads of V (lane i of a group of 16
    // reads four columns of key i / 4 and receives column i of four keys)
    const int krow = kw * S::WK + lq;
    const int ka = krow * S::RB, kx = S::swz(krow) ^ lh;   // (2 s + lh) ^ swz = 2 s ^ kx
    const int ti = lane & 15, tg = (lane >> 4) & 1;
    const int vkey = kw * S::WK + 4 * lh + (ti >> 2), vcol = 2 * tg + ((ti & 3) >> 1), vb8 = (ti & 1) * 8;

    const int kb_first = (int)((int64_t)nkb * part / sp), kb_end = (int)((int64_t)nkb * (part + 1) / sp);
    if (kb_first < kb_end) {
        issue(kb_first, 0);
        land(0);
    }
    tile_wait();
    for (int kb = kb_first; kb < kb_end; ++kb) {
        const int cur = (kb - kb_first) & 1;
        if (kb + 1 < kb_end) issue(kb + 1, cur ^ 1);
        const unsigned char* const kt = smem + cur * S::kBuf;
        const unsigned char* const vt = kt + S::kTile;
        const int key0 = kb * S::TK + kw * S::WK;
        if (key0 <= any_see) {
            // fragments of 32 keys some query sees
            const bool more = NK > 1 && key0 + 32 <= any_see;
            // S^T: lane l, register r of s[t] holds key 32 t + 8 (r / 4) + 4 lh + r % 4
            fa_f16 s[NK];
#pragma unroll
            for (int t = 0; t < NK; ++t) {
#pragma unroll
                for (int r = 0; r < 16; ++r) s[t][r] = 0.f;
                if (t > 0 && !more) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) s[t][r] = -INFINITY;
                    continue;
                }
                fa_h8 kf[HD / 16];
#pragma unroll
                for (int d = 0; d < HD / 16; ++d)
                    kf[d] = *reinterpret_cast<const fa_h8*>(kt + ka + t * 32 * S::RB + (((2 * d) ^ kx) << 4));
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int d = 0; d < HD / 16; ++d)
                    s[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[d], qf[d], s[t], 0, 0, 0);
            }
            // the values are requested before the softmax that weighs them:
            // k-slot (lh, e) of V^T holds key 16 u + 4 lh + e (e < 4) or 16 u +
            // 8 + 4 lh + e - 4 (e >= 4)
            fa_h8 vf[2][ND];
            auto values = [&](int t) {
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int j = 0; j < ND; ++j) {
                        const int c = 4 * j + vcol;
                        const int k1 = 32 * t + 16 * u + vkey, k2 = k1 + 8;
                        const unsigned char* const a1 = vt + k1 * S::RB + ((c ^ S::swz(k1)) << 4) + vb8;
                        const unsigned char* const a2 = vt + k2 * S::RB + ((c ^ S::swz(k2)) << 4) + vb8;
                        const fa_h4 lo = __builtin_bit_cast(
                            fa_h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) fa_s4*)a1));
                        const fa_h4 hi = __builtin_bit_cast(
                            fa_h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) fa_s4*)a2));
                        vf[u][j] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                    }
            };
            values(0);
            __builtin_amdgcn_sched_barrier(0);
            if (key0 + S::WK - 1 > all_see) {
#pragma unroll
                for (int t = 0; t < NK; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (key0 + 32 * t + 8 * (r >> 2) + 4 * lh + (r & 3) > last_key) s[t][r] = -INFINITY;
            }
            float mx = fmaxf(s[0][0], s[0][1]);
#pragma unroll
            for (int r = 2; r < 16 * NK; ++r) mx = fmaxf(mx, s[r / 16][r % 16]);
            mx = fa_pair_max(mx) * sl2;  // the tile's max in base-2 units (sl2 > 0)
            // v_exp_f32 flushes results below 2^-126 to zero: weights that
            // small (scores 87 natural units under the row max) are zero in
            // any FP16 / FP32 sum here anyway.
            // Lazy rescale: the running max moves only when some query's tile
            // max exceeds it by more than 8 (a factor 256; P stays <= 256,
            // well inside FP16).  A query that has seen no key yet has m =
            // -inf: its first visible tile moves it, and until then every
            // weight is exp2(-inf - finite) = 0 (nm below).
            if (__any(mx > m + 8.f)) {
                const float mnew = fmaxf(m, mx);
                const float alpha = m == mnew ? 1.f : __builtin_amdgcn_exp2f(m - mnew);
                l *= alpha;
#pragma unroll
                for (int j = 0; j < ND; ++j) o[j] *= alpha;
                m = mnew;
            }
            const float nm = m == -INFINITY ? 0.f : -m;
#pragma unroll
            for (int t = 0; t < NK; ++t) {
                if (t > 0 && !more) break;
                fa_h8 pb[2];   // B operands: 16 keys each
                float ls[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float p = __builtin_amdgcn_exp2f(fmaf(s[t][r], sl2, nm));
                    ls[r & 3] += p;
                    pb[r >> 3][r & 7] = (_Float16)p;
                }
                l += (ls[0] + ls[1]) + (ls[2] + ls[3]);
                if (t > 0) values(t);
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int j = 0; j < ND; ++j)
                        o[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[u][j], pb[u], o[j], 0, 0, 0);
            }
        }
        if (kb + 1 < kb_end) land(cur ^ 1);
        tile_wait();
    }

    // The KS wavefronts of a query each finish QW of the 4 ND quads of O^T (quad
    // x = 4 j + r / 4: four head dims of the lane's query): they hand the others'
    // quads over through LDS (the tiles are done with) and add the shares of
    // their own in wavefront order.  Left to one wavefront, the merge and the
    // stores were 0.9 of 5.0 us of the smallest calls.
    constexpr int QW = S::QW;
    fa_f4 own[QW];
    auto quad = [&](int x) {
        const fa_f16& f = o[x / 4];
        return fa_f4{f[4 * (x % 4)], f[4 * (x % 4) + 1], f[4 * (x % 4) + 2], f[4 * (x % 4) + 3]};
    };
    if constexpr (KS == 1) {
#pragma unroll
        for (int x = 0; x < QW; ++x) own[x] = quad(x);
    } else {
        fa_f4* const recs0 = reinterpret_cast<fa_f4*>(smem) + lane;
        fa_f4* const mine = recs0 + wave * S::kRec;
        if (row0 < L) {
            static_for<KS>([&](auto c) {
                constexpr int k = decltype(c)::value;
                if (kw == k) {
#pragma unroll
                    for (int x = 0; x < 4 * ND; ++x) {
                        if (x / QW == k) own[x % QW] = quad(x);
                        else mine[(x < k * QW ? x : x - QW) * 64] = quad(x);
                    }
                }
            });
            mine[(4 * ND - QW) * 64] = fa_f4{m, l, 0.f, 0.f};
        }
        __syncthreads();
        if (row0 >= L) return;
        float ms = 0.f, ls = 0.f;
        fa_f4 sum[QW];
#pragma unroll
        for (int i = 0; i < KS; ++i) {
            const fa_f4* const r = recs0 + (qw * KS + i) * S::kRec;
            const fa_f4 ml = r[(4 * ND - QW) * 64];
            fa_f4 v[QW];
#pragma unroll
            for (int x = 0; x < QW; ++x) {
                v[x] = own[x];
                if (i != kw) v[x] = r[((kw < i ? kw : kw - 1) * QW + x) * 64];
            }
            if (i == 0) {
                ms = ml[0];
                ls = ml[1];
#pragma unroll
                for (int x = 0; x < QW; ++x) sum[x] = v[x];
            } else {
                const float mnew = fmaxf(ms, ml[0]);
                const float a = ms == mnew ? 1.f : __builtin_amdgcn_exp2f(ms - mnew);
                const float b = ml[0] == mnew ? 1.f : __builtin_amdgcn_exp2f(ml[0] - mnew);
                ms = mnew;
                ls = ls * a + ml[1] * b;
#pragma unroll
                for (int x = 0; x < QW; ++x) sum[x] = sum[x] * a + v[x] * b;
            }
        }
        m = ms;
        l = ls;
#pragma unroll
        for (int x = 0; x < QW; ++x) own[x] = sum[x];
    }
    l += __shfl_xor(l, 32);
    if (row >= L) return;
    // head dim of element 0 of own quad x
    auto dim = [&](int x) { return 8 * (kw * QW + x) + 4 * lh; };
    if (sp > 1) {
        // this part's record (O, m in natural units, l); attn_combine adds them
        float* const rec = recs + (((int64_t)row * n_q + head) * sp + part) * (HD + 2);
#pragma unroll
        for (int x = 0; x < QW; ++x)
#pragma unroll
            for (int e = 0; e < 4; ++e) rec[dim(x) + e] = own[x][e];
        if (kw == 0 && lh == 0) {
            rec[HD] = m * 0.6931471805599453f;
            rec[HD + 1] = l;
        }
        return;
    }
    const float inv = 1.0f / l;
    uint16_t* const orow = out + (int64_t)row * qstride + (int64_t)head * HD;
#pragma unroll
    for (int x = 0; x < QW; ++x) {
        uint16_t h[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = f2h(own[x][e] * inv);
        u2v w;
        w.x = (uint32_t)h[0] | ((uint32_t)h[1] << 16);
        w.y = (uint32_t)h[2] | ((uint32_t)h[3] << 16);
        *reinterpret_cast<fa_any8*>(orow + dim(x)) = w;
    }
}

// One tile of up to 64 or 128 keys (the smallest calls): fragments of 16 rows, whose
// chain of S, softmax and P V is half as long as that of 32, on
// v_mfma_f32_16x16x32_f16.  A workgroup has 64 rows of one head, a wavefront 16 of
// them; K and V come by LDS-DMA (through registers where they are not on 16 bytes),
// requested with q, and are waited for once.  (K straight into the operands, by
// every wavefront, took 64 KB through the L1 of a CU: 5.4 us for 64 rows and keys.)
// What bounds it: the launch and that one memory round trip.  16 rows and keys of 16
// heads of 128 3.1 us, 64 rows and keys 4.0, 128 rows and keys 4.9; fa_kernel 4.8, 5.9
// and 6.5, the 16-row fragments with K and V staged through registers 4.1, 5.1 and 6.9.
constexpr int kOneTile = 128;

template <int HD, int NT, bool AL>
__global__ __launch_bounds__(kFaThreads, 2) void fa_one_tile_kernel(const uint16_t* __restrict__ q,
                                                                   const uint16_t* __restrict__ Kc,
                                                                   const uint16_t* __restrict__ Vc, int L, int valid_len,
                                                                   int n_q, int n_kv, int bidir,
                                                                   uint16_t* __restrict__ out) {
    using S = FaShape<HD, 1, 2>;   // the layout of a key row
    constexpr int ND = HD / 16, kTile = 16 * NT * S::RB, P = 16 * NT / S::RPC / 4;
    __shared__ __align__(1024) unsigned char tiles[2 * kTile];   // K, then V
    const unsigned char* const vt = tiles + kTile;
    const int rt = (int)blockIdx.x, head = (int)blockIdx.y, g = head / (n_q / n_kv);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lq = lane & 15, lg = lane >> 4;
    const int64_t qstride = (int64_t)n_q * HD, kvstride = (int64_t)n_kv * HD;
    const int row0 = 64 * rt + 16 * wave, row = row0 + lq, p0 = valid_len - L;
    const int last_key = bidir ? valid_len - 1 : min(p0 + row, valid_len - 1);
    const int any_see = bidir ? valid_len - 1 : min(p0 + row0 + 15, valid_len - 1);

    // q rows: B operand, lane l holds query l % 16, d 32 s + 8 (l / 16) ..
    fa_h8 qf[HD / 32];
    {
        const uint16_t* const qrow = q + (int64_t)min(row, L - 1) * qstride + (int64_t)head * HD + 8 * lg;
#pragma unroll
        for (int d = 0; d < HD / 32; ++d)
            qf[d] = __builtin_bit_cast(fa_h8, (u4v)*reinterpret_cast<const fa_any16*>(qrow + 32 * d));
    }
    // wavefront w copies rows RPC (w P + j) .. of the tile; keys past the end repeat
    // the last one
    const unsigned char* const kb0 = reinterpret_cast<const unsigned char*>(Kc + (int64_t)g * HD);
    const unsigned char* const vb0 = reinterpret_cast<const unsigned char*>(Vc + (int64_t)g * HD);
    const uint32_t dst = __builtin_amdgcn_readfirstlane(lds_addr(tiles) + wave * P * 1024);
    u4v reg[AL ? 1 : 2 * P];
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const int r = S::RPC * (wave * P + j) + lane / S::CH;
        const uint32_t off = (uint32_t)min(r, valid_len - 1) * (uint32_t)(kvstride * 2) +
                             (uint32_t)(((lane % S::CH) ^ S::swz(r)) * 16);
        if constexpr (AL) {
            dma16(off, kb0, dst + j * 1024);
            dma16(off, vb0, dst + kTile + j * 1024);
        } else {
            reg[2 * j] = *reinterpret_cast<const fa_any16*>(kb0 + off);
            reg[2 * j + 1] = *reinterpret_cast<const fa_any16*>(vb0 + off);
        }
    }
    if constexpr (!AL) {
#pragma unroll
        for (int j = 0; j < 2 * P; ++j)
            *reinterpret_cast<u4v*>(tiles + (j & 1) * kTile + (wave * P + j / 2) * 1024 + lane * 16) = reg[j];
    }
    wait_vm_barrier<0>();
    if (row0 >= L) return;

    // S^T: lane l, register r of s[t] holds key 16 t + 4 (l / 16) + r of query l % 16
    fa_f4 s[NT];
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        s[t] = fa_f4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        if (16 * t <= any_see) {
            s[t] = fa_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int d = 0; d < HD / 32; ++d) {
                const int k = 16 * t + lq;   // A operand: lane l holds key l % 16, the same d
                const fa_h8 kf = *reinterpret_cast<const fa_h8*>(tiles + k * S::RB + (((4 * d + lg) ^ S::swz(k)) << 4));
                s[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[d], s[t], 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (16 * t + 4 * lg + r > last_key) s[t][r] = -INFINITY;
                mx = fmaxf(mx, s[t][r]);
            }
        }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    const float sl2 = 1.4426950408889634f / sqrtf((float)HD);
    const float m = fmaxf(mx, __shfl_xor(mx, 32)) * sl2, nm = m == -INFINITY ? 0.f : -m;
    float l = 0.f;
    fa_h8 pb[NT / 2];   // B operands of 32 keys: 16 of one fragment and 16 of the next
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float p = __builtin_amdgcn_exp2f(fmaf(s[t][r], sl2, nm));
            l += p;
            pb[t / 2][4 * (t % 2) + r] = (_Float16)p;
        }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);

    // O^T: d = 16 j + 4 (l / 16) + r of query l % 16
    const int tkey = 4 * lg + (lq >> 2), tcol = (lq & 3) >> 1, tb = (lq & 1) * 8;
    fa_f4 o[ND];
#pragma unroll
    for (int j = 0; j < ND; ++j) o[j] = fa_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < NT / 2; ++u) {
        if (32 * u > any_see) break;
#pragma unroll
        for (int j = 0; j < ND; ++j) {
            const int c = 2 * j + tcol, k1 = 32 * u + tkey, k2 = k1 + 16;
            const unsigned char* const a1 = vt + k1 * S::RB + ((c ^ S::swz(k1)) << 4) + tb;
            const unsigned char* const a2 = vt + k2 * S::RB + ((c ^ S::swz(k2)) << 4) + tb;
            const fa_h4 lo = __builtin_bit_cast(
                fa_h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) fa_s4*)a1));
            const fa_h4 hi = __builtin_bit_cast(
                fa_h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) fa_s4*)a2));
            o[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), pb[u],
                                                          o[j], 0, 0, 0);
        }
    }
    if (row >= L) return;
    const float inv = 1.0f / l;
    uint16_t* const orow = out + (int64_t)row * qstride + (int64_t)head * HD + 4 * lg;
#pragma unroll
    for (int j = 0; j < ND; ++j) {
        u2v w;
        w.x = (uint32_t)f2h(o[j][0] * inv) | ((uint32_t)f2h(o[j][1] * inv) << 16);
        w.y = (uint32_t)f2h(o[j][2] * inv) | ((uint32_t)f2h(o[j][3] * inv) << 16);
        *reinterpret_cast<fa_any8*>(orow + 16 * j) = w;
    }
}

template <int HD, bool AL>
int fa_one_tile_launch(const uint16_t* q, const uint16_t* Kc, const uint16_t* Vc, int L, int valid_len, int n_q,
                       int n_kv, int bidir, uint16_t* out, hipStream_t st) {
    const dim3 grid((unsigned)((L + 63) / 64), (unsigned)n_q);
    if (valid_len <= 64)
        fa_one_tile_kernel<HD, 4, AL><<<grid, kFaThreads, 0, st>>>(q, Kc, Vc, L, valid_len, n_q, n_kv, bidir, out);
    else
        fa_one_tile_kernel<HD, 8, AL><<<grid, kFaThreads, 0, st>>>(q, Kc, Vc, L, valid_len, n_q, n_kv, bidir, out);
    return launch_check("attention (one tile)");
}

template <int HD, int KS, int NK, bool AL>
int fa_launch(const uint16_t* q, const uint16_t* Kc, const uint16_t* Vc, int L, int valid_len, int n_q, int n_kv,
              int bidir, int gb, int sp, float* recs, uint16_t* out, hipStream_t st) {
    using S = FaShape<HD, KS, NK>;
    const int rows = 32 * (4 / KS / gb);
    const int64_t blocks = (int64_t)((L + rows - 1) / rows) * n_kv * (n_q / n_kv / gb) * sp;
    if (blocks > (1 << 30) || n_kv > 65535) return fail(BX_EINVAL, "attention: too many heads");
    const int cus = num_cus();
    const int mirror = !bidir && sp == 1 && blocks > cus && blocks <= 2 * cus ? cus : (int)blocks;
    const void* fn = reinterpret_cast<const void*>(&fa_kernel<HD, KS, NK, AL>);
    if constexpr (S::kLds > 64 * 1024) {
        static std::atomic<uint64_t> allowed{0};
        if (int rc = allow_lds(allowed, fn, S::kLds, "attention: LDS attribute")) return rc;
    }
    fa_kernel<HD, KS, NK, AL><<<dim3((unsigned)blocks), kFaThreads, S::kLds, st>>>(q, Kc, Vc, L, valid_len, n_q, n_kv, bidir,
                                                                         gb, mirror, sp, recs, out);
    if (int rc = launch_check("attention (mfma)")) return rc;
    return sp > 1 ? attn_combine(recs, n_q, L, HD, sp, out, st) : BX_OK;
}

// Key shares per workgroup (KS) and heads sharing a tile (gb), from the number
// of (32 rows, head) fragments against the CUs: one fragment per wavefront
// where they fill two workgroups per CU (2048 causal rows, 32 heads: KS 1 52
// us, KS 2 55), two wavefronts a fragment below that (2000 rows, 16 heads: KS
// 2 31.5 us, KS 1 42.6, KS 4 51), four where they leave CUs idle and the walk
// over the keys is what takes the time (500 rows bidirectional, 16 heads: KS 4
// 9.3 us, KS 2 11.5, KS 1 15.3).  Fewer fragments still over long caches:
// `sp` workgroups share the keys, as many as the caller's workspace has
// records for, and a second launch merges them (64 rows after 2000 keys, 16
// heads: 12 us, one workgroup to all keys 21.9).
template <int HD, bool AL>
int fa_dispatch(const uint16_t* q, const uint16_t* Kc, const uint16_t* Vc, int L, int valid_len, int n_q, int n_kv,
                int bidir, void* ws, uint16_t* out, hipStream_t st) {
    const int G = n_q / n_kv, cus = num_cus();
    const int64_t frags = (int64_t)((L + 31) / 32) * n_q;
    float* const recs = static_cast<float*>(ws);
    // 128 keys in 64 KB: two workgroups a CU, more rounds of them cost more than
    // 32-row fragments (2048 rows of 32 heads 14.6 us against 14.0; of 16 heads 7.9
    // against 10.2)
    if (n_q <= 65535 &&
        (valid_len <= 64 || (valid_len <= kOneTile && (int64_t)((L + 63) / 64) * n_q <= 2 * cus)))
        return fa_one_tile_launch<HD, AL>(q, Kc, Vc, L, valid_len, n_q, n_kv, bidir, out, st);
    if (frags <= cus && valid_len > 256) {
        const int tiles = (valid_len + 127) / 128, room = attn_ws_splits(L, valid_len);
        int sp = (int)std::min<int64_t>({cus / frags, room, tiles / 2});
        // a tile takes 1.1 us, the second launch about 4
        if (sp < 2 || (tiles - tiles / sp) * 1.1 < 4.5) sp = 1;
        return fa_launch<HD, 4, 1, AL>(q, Kc, Vc, L, valid_len, n_q, n_kv, bidir, 1, sp, recs, out, st);
    }
    if (frags <= 4 * cus) {
        const int gb = G % 2 == 0 && frags > 2 * cus ? 2 : 1;
        return fa_launch<HD, 2, 1, AL>(q, Kc, Vc, L, valid_len, n_q, n_kv, bidir, gb, 1, recs, out, st);
    }
    const int gb = G % 4 == 0 ? 4 : G % 2 == 0 ? 2 : 1;
    return fa_launch<HD, 1, 2, AL>(q, Kc, Vc, L, valid_len, n_q, n_kv, bidir, gb, 1, recs, out, st);
}

}  // namespace

bool attn_mfma_supported(int L, int hd, float softcap, int window, const float* mask) {
    return L >= 16 && (hd == 64 || hd == 128) && softcap == 0.f && window <= 0 && mask == nullptr;
}

int attn_mfma(const uint16_t* q, const uint16_t* Kc, const uint16_t* Vc, int L, int valid_len, int n_q, int n_kv,
              int hd, int bidir, void* ws, uint16_t* out, hipStream_t st) {
    const bool al = ((reinterpret_cast<uintptr_t>(Kc) | reinterpret_cast<uintptr_t>(Vc)) & 15) == 0;
    const auto run = hd == 128 ? (al ? fa_dispatch<128, true> : fa_dispatch<128, false>)
                               : (al ? fa_dispatch<64, true> : fa_dispatch<64, false>);
    return run(q, Kc, Vc, L, valid_len, n_q, n_kv, bidir, ws, out, st);
}

}  // namespace bx
