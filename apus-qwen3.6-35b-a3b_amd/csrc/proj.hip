// proj.hip -- the bf16 projections on either side of the attention path
// (c/bf16.h:178-231: y[m][o] = rnd(sum_k w[o][k] x[m][k]), w [O][K],
// x [M][K], y [M][O], bf16 codes in and out, fp32 accumulation), the
// reference's apus_bf16_gemv_hot / apus_bf16_gemm_hot and the
// ApusBackendHooks bf16_gemv / bf16_gemm slots (c/backend_metal.h:68-75).
//
// The kernels:
//   k_gemm_seq   one lane per output, the k sum in the reference's order
//                (ascending, one rounding per multiply and per add: the
//                scalar anchor c/bf16.h:285-293, which the reference's
//                threaded and Metal paths reproduce bitwise). Bitwise
//                against the reference (products below fp32's normal range
//                aside: see k_gemm_seq). The weight row is read 16 bytes
//                at a time, 16 to 32 pieces ahead of the add chain; the x row
//                is staged in LDS once per wavefront.
//   k_gemm_seq64 the same chains (K a multiple of 64), the weights streamed
//                and widened into LDS by wavefronts of their own for up to
//                four rows at a time.
//   k_gemm_tile  the 32x32x16 bf16 MFMA with fp32 accumulation, for every
//                row count: a workgroup computes a (BO outputs x BM rows)
//                tile, its operands copied global -> LDS by buffer_load ...
//                lds in stages of 32 k through a 4-deep ring; each
//                wavefront reads the next k16 step's fragments while the
//                current step's MFMAs issue.
//   k_gemm_wide  the same product with one wavefront per SIMD, for calls
//                with enough tiles to fill the chip. The tile shape (and
//                with it the kernel) is the one with the least estimated
//                time; every shape accumulates an element's k16 steps in
//                the same order. The MFMA kernels sum in their own order:
//                the tolerance class of the attention kernels (|c - r| <=
//                2e-3 (|r| + esc), esc = sum_k |w x|).
// Host-pointer drop-ins keep device copies of the weights keyed by their
// host address, as the reference's Metal backend keys weights by stable
// pointers (c/backend_metal.h:42-48).
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <type_traits>
#include <unordered_map>

#include "../../include/apus_hip.h"
#include "apus_dev.h"
#include "apus_host.h"
#include "proj.h"

using namespace apus;

namespace {

typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// One output per lane: outputs blockIdx.x*64 + lane of row blockIdx.y.
// VEC: K is a multiple of 8 and the rows are 16-byte aligned. XF: the x
// row is staged in LDS as fp32 (widened once per wavefront instead of once
// per output; K up to 16384), so a k costs the weight's widening and one
// fused multiply-add. The product of two bf16 values (8-bit significands)
// is exact in fp32 whenever it lies in fp32's normal range, so the fused
// form rounds exactly where the reference's multiply-then-add does: once,
// at the add. Only a product below 2^-126 in magnitude (a subnormal,
// which the reference rounds before adding) can differ, and then only if
// the running sum is itself that small. (25.4 -> 21.0 us for 12352 x 2048.)
template <bool VEC, bool XF = false>
__global__ __launch_bounds__(64) void k_gemm_seq(const uint16_t *__restrict__ w,
                                                 const uint16_t *__restrict__ x,
                                                 uint16_t *__restrict__ y, int O, int K) {
    const int o = blockIdx.x * 64 + threadIdx.x;
    const int m = blockIdx.y;
    const uint16_t *xr = x + (size_t)m * K;
    const uint16_t *wr = w + (size_t)min(o, O - 1) * K;
    float acc = 0.0f;
    if (VEC) {
        // the x row in LDS (dynamic, K codes): its reads wait on the LDS
        // counter, so the vector-memory waits count weight loads only
        extern __shared__ __attribute__((aligned(16))) u16x8 xs_lds[];
        const int n8 = K / 8;
        if (XF) {
            float4 *xf = reinterpret_cast<float4 *>(xs_lds);
            for (int i = threadIdx.x; i < n8; i += 64) {
                const u16x8 v = reinterpret_cast<const u16x8 *>(xr)[i];
                xf[2 * i] = make_float4(bf2f(v[0]), bf2f(v[1]), bf2f(v[2]), bf2f(v[3]));
                xf[2 * i + 1] = make_float4(bf2f(v[4]), bf2f(v[5]), bf2f(v[6]), bf2f(v[7]));
            }
        } else {
            for (int i = threadIdx.x; i < n8; i += 64)
                xs_lds[i] = reinterpret_cast<const u16x8 *>(xr)[i];
        }
        __syncthreads();
        // k values 8i .. 8i+7 of x as floats
        auto xk = [&](int i, float (&f)[8]) {
            if (XF) {
                const float4 *xf = reinterpret_cast<const float4 *>(xs_lds);
                const float4 a = xf[2 * i], b = xf[2 * i + 1];
                f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
                f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
            } else {
                const u16x8 v = xs_lds[i];
#pragma unroll
                for (int j = 0; j < 8; j++) f[j] = bf2f(v[j]);
            }
        };
        const u16x8 *w8 = reinterpret_cast<const u16x8 *>(wr);
        constexpr int R = 16;          // pieces per round; two register sets
        // rounds alternate between the sets: while one set is summed the
        // next round's loads are in flight into the other. Prefetch indices
        // are clamped to the row (no branch around a load), so each wait
        // counts only the loads issued after the set it needs.
        u16x8 qa[R], qb[R];
#pragma unroll
        for (int i = 0; i < R; i++) qa[i] = w8[min(i, n8 - 1)];
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        int p = 0;
        for (; p + 2 * R <= n8; p += 2 * R) {
#pragma unroll
            for (int i = 0; i < R; i++) qb[i] = w8[min(p + R + i, n8 - 1)];
            // keep the prefetches here (the compiler would sink each load
            // to its first use and wait on it there)
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < R; i++) {
                float xv[8];
                xk(p + i, xv);
#pragma unroll
                for (int j = 0; j < 8; j++) acc = fmaf(bf2f(qa[i][j]), xv[j], acc);
            }
#pragma unroll
            for (int i = 0; i < R; i++) qa[i] = w8[min(p + 2 * R + i, n8 - 1)];
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < R; i++) {
                float xv[8];
                xk(p + R + i, xv);
#pragma unroll
                for (int j = 0; j < 8; j++) acc = fmaf(bf2f(qb[i][j]), xv[j], acc);
            }
        }
        for (int i = 0; p + i < n8; i++) {
            const u16x8 wv = w8[p + i];
            float xv[8];
            xk(p + i, xv);
#pragma unroll
            for (int j = 0; j < 8; j++) acc = fmaf(bf2f(wv[j]), xv[j], acc);
        }
    } else {
        for (int k = 0; k < K; k++) acc = acc + bf2f(wr[k]) * bf2f(xr[k]);
    }
    if (o < O) y[(size_t)m * O + o] = f2bf(acc);
}

// The same sums for K a multiple of 64 (up to 16384): 64 outputs of R rows
// (1 .. 4) a workgroup. Wavefront r < R runs row r's 64 chains, a lane each,
// and four more stream the weights for all rows, widen them and lay them in
// LDS as the chains read them. In k_gemm_seq a wavefront does all of this
// for one row, so that a k costs it 2.5 instructions besides the wait for
// the sum before it, its loads are 16-byte pieces of 64 rows, and the weights
// are read once per row. 12352 x 2048: one row 18.0 -> 16.3 us, 3 rows 30.2 ->
// 19.5, 8 rows 72 -> 31; 2048 x 4096 33.1 -> 27.2. What is left is the chain:
// 6 ns a k, where a dependent add alone takes 4 and each chunk adds its
// barrier and the wait for its first reads (reads placed between the
// multiply-adds, or a part ahead of them, made it 6.5 to 6.9).
constexpr int kSeqK = 64;                  // k per chunk
constexpr int kSeqDepth = 8;               // chunks in flight per loader
__global__ __launch_bounds__(512) void k_gemm_seq64(const uint16_t *__restrict__ w,
                                                    const uint16_t *__restrict__ x,
                                                    uint16_t *__restrict__ y, int M, int O, int K,
                                                    int R) {
    // chunk buffers [k / 4][row][4] (PITCH: 16 rows of padding spread a
    // loader's 8 pieces of a row over the banks), then x as fp32
    constexpr int PITCH = 64 * 4 + 4;
    __shared__ __attribute__((aligned(16))) float wl[2][(kSeqK / 4) * PITCH];
    extern __shared__ __attribute__((aligned(16))) float4 xf[];
    const int m0 = blockIdx.y * R, o0 = blockIdx.x * 64, nch = K / kSeqK;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int e = threadIdx.x; e < R * (K / 8); e += 64 * (4 + R)) {   // x rows (past M: the last)
        const int r = e / (K / 8), i = e % (K / 8);
        const u16x8 v = reinterpret_cast<const u16x8 *>(x + (size_t)min(m0 + r, M - 1) * K)[i];
        xf[2 * e] = make_float4(bf2f(v[0]), bf2f(v[1]), bf2f(v[2]), bf2f(v[3]));
        xf[2 * e + 1] = make_float4(bf2f(v[4]), bf2f(v[5]), bf2f(v[6]), bf2f(v[7]));
    }
    if (wave >= R) {
        // loader: rows r0 + lane / 8 and that + 8, 16-byte piece lane % 8 of
        // each chunk's 128 bytes. Loads past the last chunk read it again.
        const int r0 = (wave - R) * 16 + (lane >> 3), pc = lane & 7;
        const u16x8 *src[2];
#pragma unroll
        for (int i = 0; i < 2; i++)
            src[i] = reinterpret_cast<const u16x8 *>(w + (size_t)min(o0 + r0 + 8 * i, O - 1) * K) + pc;
        u16x8 q[kSeqDepth][2];
        auto load = [&](int c, u16x8 (&d)[2]) {
#pragma unroll
            for (int i = 0; i < 2; i++) d[i] = src[i][min(c, nch - 1) * (kSeqK / 8)];
        };
        auto put = [&](int c, const u16x8 (&d)[2]) {
#pragma unroll
            for (int i = 0; i < 2; i++) {
                float *p = wl[c & 1] + 2 * pc * PITCH + (r0 + 8 * i) * 4;
                *reinterpret_cast<float4 *>(p) = make_float4(bf2f(d[i][0]), bf2f(d[i][1]), bf2f(d[i][2]), bf2f(d[i][3]));
                *reinterpret_cast<float4 *>(p + PITCH) = make_float4(bf2f(d[i][4]), bf2f(d[i][5]), bf2f(d[i][6]), bf2f(d[i][7]));
            }
        };
#pragma unroll
        for (int c = 0; c < kSeqDepth; c++) load(c, q[c]);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        for (int c0 = 0; c0 < nch; c0 += kSeqDepth) {
#pragma unroll
            for (int j = 0; j < kSeqDepth; j++) {
                const int c = c0 + j;
                if (c < nch) {
                    // (this buffer's readers passed the barrier of chunk c - 1)
                    put(c, q[j]);
                    load(c + kSeqDepth, q[j]);
                    // keep the loads here (they would be sunk to their use)
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_sched_barrier(0);
                    __syncthreads();               // chunk c is in place
                }
            }
        }
        return;
    }
    const float4 *xc = xf + wave * (K / 4);
    float acc = 0.0f;
    for (int c = 0; c < nch; c++) {
        __syncthreads();                           // chunk c is in place
        const float4 *wc = reinterpret_cast<const float4 *>(wl[c & 1]) + lane;
#pragma unroll
        for (int i = 0; i < kSeqK / 4; i++) {
            const float4 a = wc[i * (PITCH / 4)], b = xc[c * (kSeqK / 4) + i];
            acc = fmaf(a.x, b.x, acc);
            acc = fmaf(a.y, b.y, acc);
            acc = fmaf(a.z, b.z, acc);
            acc = fmaf(a.w, b.w, acc);
        }
    }
    const int m = m0 + wave;
    if (m < M && o0 + lane < O) y[(size_t)m * O + o0 + lane] = f2bf(acc);
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pk2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
int check_dims(size_t M, size_t O, size_t K) {
    if (M > 0x7fffffffu || O > 0x7fffffffu || K > 0x7fffffffu)
        return set_error(kErrUnsupported, "gemm dims past 2^31");
    return kOk;
}

// byte offset of 16-byte chunk c (0..3) of row r in a stage's 64-byte rows:
// chunks are XOR-swizzled by (r / 4) % 4, so the 32 rows one MFMA operand
// read touches spread over the LDS banks
__device__ __forceinline__ int tile_slot(int r, int c) { return r * 64 + ((c ^ ((r >> 2) & 3)) << 4); }

constexpr int kTileStages = 4;            // LDS ring depth (stages of 32 k)

// Workgroup -> (output tile, row tile). Workgroups are dealt round-robin
// to the 8 XCDs (id % 8), each XCD running its ids in order, so XCD x gets
// tiles x q .. x q + q - 1 (q an eighth of the tiles) of an order in which
// the 32 tiles that an XCD runs together share operand tiles, which stay in
// that XCD's L2 while they walk K in step: with 8 or more row tiles, blocks
// of 4 output x 8 row tiles (12 distinct operand tiles instead of 18 with
// whole row-tile columns); with fewer, an output tile's row tiles one after
// the other. Every XCD has the same number of tiles to within one (whole
// 4 x 8 blocks dealt to XCDs left half of the chip idle below 8 blocks:
// 2048 outputs x 512 rows, K = 4096, 34.7 us, now 17.4).
__host__ __device__ inline int tile_grid(int nbo, int nbm) { return (nbo * nbm + 7) / 8 * 8; }
__host__ __device__ inline void tile_of(int id, int nbo, int nbm, int &ob, int &mb) {
    const int n = nbo * nbm, q = (n + 7) / 8, t = (id % 8) * q + id / 8;
    if (t >= n) {
        ob = nbo;                                  // past the last tile
        mb = 0;
        return;
    }
    if (nbm < 8) {
        ob = t / nbm;
        mb = t % nbm;
        return;
    }
    // bands of 8 row tiles; in a band, blocks of 4 output tiles, row fastest
    const int band = t / (8 * nbo), rows = min(8, nbm - 8 * band);
    const int p = t - 8 * nbo * band;
    const int blk = p / (4 * rows), w = min(4, nbo - 4 * blk), e = p - 4 * rows * blk;
    ob = 4 * blk + e % w;
    mb = 8 * band + e / w;
}

__device__ __forceinline__ int seg_of(const GemmSegs &g, int o) {
    int i = 0;
#pragma unroll
    for (int j = 1; j < kMaxSegs; j++)
        if (j < g.n && o >= g.row0[j]) i = j;
    return i;
}

// bf16 stores of a wavefront's TO x TMM accumulator tiles (D[o][m]): tile
// (t, u) holds outputs ob0 + 32 t .. and rows mb0 + 32 u + lane % 32; lane
// -> o = 8 (i / 4) + 4 (lane / 32) + i % 4 of register i. Each 32-output
// tile lies in one segment.
template <int TO, int TMM>
__device__ __forceinline__ void store_tiles(const GemmSegs &sg, const f32x16 (&acc)[TO][TMM],
                                            int ob0, int mb0, int O, int M, int lane) {
#pragma unroll
    for (int t = 0; t < TO; t++) {
        const int ot = ob0 + t * 32;
        if (ot >= O) continue;
        const int si = seg_of(sg, ot);
        uint16_t *yb = sg.y[si] - sg.row0[si];
        const int ld = sg.ldy[si];
        const bool vec = ((ld | sg.row0[si]) & 3) == 0 && ((uintptr_t)sg.y[si] & 7) == 0;
#pragma unroll
        for (int u = 0; u < TMM; u++) {
            const int m = mb0 + u * 32 + (lane & 31);
            if (m >= M) continue;
            const f32x16 &a = acc[t][u];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int o = ot + 8 * q + 4 * (lane >> 5);
                if (vec) {
                    if (o < O)
                        *reinterpret_cast<uint2 *>(yb + (size_t)m * ld + o) =
                            make_uint2(pk2(a[4 * q], a[4 * q + 1]), pk2(a[4 * q + 2], a[4 * q + 3]));
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (o + i < O) yb[(size_t)m * ld + o + i] = f2bf(a[4 * q + i]);
                }
            }
        }
    }
}

// y[m][o] = rnd(sum_k w[o][k] x[m][k]) on the 32x32x16 bf16 MFMA. The
// workgroup has WO x WM wavefronts; wavefront (wo, wm) = (wave / WM,
// wave % WM) -- so the WM wavefronts sharing output columns sit on
// different SIMDs -- computes TO x TMM MFMA tiles: outputs
// o0 + 32 (TO wo + t) .., rows m0 + 32 (TMM wm + u) ... The product is
// formed transposed (D[o][m]: A = w rows, B = x rows) so that a lane holds
// 4 consecutive outputs of one row and stores them as 8 bytes.
// Stages: each stage's w rows (BO x 64 B) and x rows (BM x 64 B) are copied
// global -> LDS in 1 KiB pieces (16 rows each; lane L fills byte 16 L of
// the piece: row L / 4, chunk (L % 4) ^ ((row / 4) % 4)); rows past O or M
// lie past their buffer's end and read zero. Stage s is issued ST - 1
// stages ahead, unconditionally (past the last stage the copy re-reads
// it), so every wait is a constant count; one barrier per stage. MFMAs of
// tiles wholly past O or M are skipped (wave-uniform).
// Workgroup order: the row tiles of an output tile are dealt to one XCD
// (block ids congruent mod 8), so they share its w rows in that XCD's L2.
// Split K (part != nullptr): block b works on k stages of split b / nb
// (nb: the blocks of one split) and stores its fp32 partial tile to
// part[split][m][o]; k_gemm_reduce then sums the splits in order.
template <int WO, int WM, int TO, int TMM, int ST>
__global__ __launch_bounds__(64 * WO * WM) void k_gemm_tile(GemmSegs sg,
                                                       const uint16_t *__restrict__ x, int M,
                                                       int K, float *__restrict__ part, int nsplit) {
    const int O = sg.row0[sg.n];
    constexpr int NW = WO * WM, BO = 32 * TO * WO, BM = 32 * TMM * WM;
    constexpr int PB = BO * 64, SB = (BO + BM) * 64;
    constexpr int NPIECE = (BO + BM) / 16;
    static_assert(NPIECE % NW == 0, "copy pieces must split evenly over the wavefronts");
    constexpr int PPW = NPIECE / NW;
    __shared__ __attribute__((aligned(16))) char sm[ST * SB];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wo = wave / WM, wm = wave % WM;
    const int nbo = (O + BO - 1) / BO, nbm = (M + BM - 1) / BM;
    const int nb = tile_grid(nbo, nbm);
    const int id = blockIdx.x % nb, ks = blockIdx.x / nb;
    int ob, mb;
    tile_of(id, nbo, nbm, ob, mb);
    if (ob >= nbo || mb >= nbm) return;         // (the grid rounds up to whole groups)
    const int o0 = ob * BO, m0 = mb * BM;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_void *)sm);
    // this wave's copy pieces: the buffer of each (x, or its weight
    // segment; wave-uniform) and each lane's byte offset in it
    i32x4 rs[PPW];
    int voff[PPW];
    uint32_t loff[PPW];
#pragma unroll
    for (int i = 0; i < PPW; i++) {
        const int p = wave * PPW + i;
        const bool pw = p < BO / 16;
        const int pr = pw ? p : p - BO / 16;
        const int r = pr * 16 + lane / 4;
        const int c = (lane & 3) ^ ((r >> 2) & 3);
        if (pw) {
            const int si = __builtin_amdgcn_readfirstlane(seg_of(sg, o0 + pr * 16));
            const int rows = sg.row0[si + 1] - sg.row0[si], gr = o0 + r - sg.row0[si];
            rs[i] = dma_rsrc(sg.w[si], (uint32_t)((size_t)rows * K * 2));
            voff[i] = gr < rows ? (gr * K + c * 8) * 2 : 0x7fffffff;
        } else {
            rs[i] = dma_rsrc(x, (uint32_t)((size_t)M * K * 2));
            voff[i] = m0 + r < M ? ((m0 + r) * K + c * 8) * 2 : 0x7fffffff;
        }
        loff[i] = pw ? pr * 1024 : PB + pr * 1024;
    }
    // this block's k stages: [kt0, kt0 + nk)
    const int nkall = K / 32;
    const int kt0 = ks * nkall / nsplit, nk = (ks + 1) * nkall / nsplit - kt0;
    auto issue = [&](int st) {
        const int kb = (kt0 + min(st, nk - 1)) * 64;
        const uint32_t base = lds0 + (st % ST) * SB;
#pragma unroll
        for (int i = 0; i < PPW; i++) dma16(rs[i], voff[i], kb, base + loff[i]);
    };
    f32x16 acc[TO][TMM];
#pragma unroll
    for (int t = 0; t < TO; t++)
#pragma unroll
        for (int u = 0; u < TMM; u++) acc[t][u] = f32x16{};
    auto rd = [&](int kt, int s, bf16x8 (&af)[TO], bf16x8 (&bf)[TMM]) {
        const char *Wl = sm + (kt % ST) * SB;
        const char *Xl = Wl + PB;
        const int c = s * 2 + (lane >> 5);
#pragma unroll
        for (int t = 0; t < TO; t++)
            af[t] = *reinterpret_cast<const bf16x8 *>(Wl + tile_slot(wo * TO * 32 + t * 32 + (lane & 31), c));
#pragma unroll
        for (int u = 0; u < TMM; u++)
            bf[u] = *reinterpret_cast<const bf16x8 *>(Xl + tile_slot(wm * TMM * 32 + u * 32 + (lane & 31), c));
    };
    const int tv = min(TO, max(0, (O - (o0 + wo * TO * 32) + 31) / 32));
    const int uv = min(TMM, max(0, (M - (m0 + wm * TMM * 32) + 31) / 32));
    // MFMAs of tiles past O or M are skipped; a wavefront whose tiles are
    // all inside runs the loop without the per-MFMA tests (as uniform
    // branches they split the loop into a block per MFMA and cost ~10 %)
    auto loop = [&](auto edge) {
        auto mma = [&](const bf16x8 (&af)[TO], const bf16x8 (&bf)[TMM]) {
#pragma unroll
            for (int t = 0; t < TO; t++)
#pragma unroll
                for (int u = 0; u < TMM; u++)
                    if (!decltype(edge)::value || (t < tv && u < uv))
                        acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[t], bf[u], acc[t][u], 0, 0, 0);
        };
#pragma unroll
        for (int s = 0; s < ST - 1; s++) issue(s);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PPW * (ST - 2)) : "memory");
        __syncthreads();
        issue(ST - 1);
        bf16x8 fa0[TO], fb0[TMM], fa1[TO], fb1[TMM];
        rd(0, 0, fa0, fb0);
        // the scheduling barriers keep each phase's LDS reads ahead of the
        // MFMAs that do not need them (left free, the scheduler sank them
        // to their first use)
        for (int kt = 0; kt < nk; kt++) {
            rd(kt, 1, fa1, fb1);
            __builtin_amdgcn_sched_barrier(0);
            mma(fa0, fb0);
            __builtin_amdgcn_sched_barrier(0);
            // stage kt+1 landed (this wave's copies), then visible to all;
            // every wave is past its reads of stage kt, whose slot the next
            // issue fills
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PPW * (ST - 2)) : "memory");
            __syncthreads();
            issue(kt + ST);
            rd(kt + 1, 0, fa0, fb0);
            __builtin_amdgcn_sched_barrier(0);
            mma(fa1, fb1);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (tv == TO && uv == TMM)
        loop(std::false_type{});
    else
        loop(std::true_type{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // D[o][m]: lane -> m = lane % 32, o = 8 (i / 4) + 4 (lane / 32) + i % 4;
    // each 32-output tile lies in one segment
    if (part) {                                 // fp32 partials, [split][m][O]
        float *pb = part + (size_t)ks * M * O;
#pragma unroll
        for (int t = 0; t < TO; t++) {
            const int ot = o0 + wo * TO * 32 + t * 32;
            if (ot >= O) continue;
#pragma unroll
            for (int u = 0; u < TMM; u++) {
                const int m = m0 + wm * TMM * 32 + u * 32 + (lane & 31);
                if (m >= M) continue;
                const f32x16 &a = acc[t][u];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int o = ot + 8 * q + 4 * (lane >> 5);
                    if (o < O)
                        *reinterpret_cast<float4 *>(pb + (size_t)m * O + o) =
                            make_float4(a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]);
                }
            }
        }
        return;
    }
    store_tiles<TO, TMM>(sg, acc, o0 + wo * TO * 32, m0 + wm * TMM * 32, O, M, lane);
}

// ---- k_gemm_wide ---------------------------------------------------------
// The same product, operands and summation order as k_gemm_tile (bitwise
// the same result), with 4 wavefronts (2 x 2), one per SIMD, of TO x TMM
// MFMA tiles each. What bounded k_gemm_tile at 256 x 256 (8 wavefronts of
// 4 x 2 tiles, 32-k stages) and what changed here, on a 2048 x 8192 x 4096
// product, 256 tiles, in us per 32 k (the MFMAs alone: 0.59):
//   0.95  as it was. 64-byte half lines per row and copy, and a wavefront
//         reads 6 fragments from LDS for 8 MFMAs;
//   0.87  4 x 4 tiles (8 reads for 16 MFMAs), 64-k stages, so that a copy
//         reads whole 128-byte lines;
//   0.77  each line touched once per XCD a stage before its copies: the
//         workgroups of an XCD walk K in step, so each stage's lines all
//         missed L2 together, and a stage was a trip to HBM long.
// The stores of a tile go through LDS as whole rows (what a call takes
// besides its k steps: 23 -> 7 us). 4096 x 12352 x 2048: 236 -> 201 us (1.03
// PFLOP/s).
// The ring holds ST stages. Three where a CU has LDS for them beside the
// fewer products of a small tile, which a copy of one stage outlasts
// (325 x 12352 x 2048, 194 workgroups of 128 x 192: two stages 29.3 us, three
// 25.6; four, at 128 x 128, no further gain), two for 256-wide tiles, and
// for 128 x 128 where two workgroups share a CU (640 x 12352: 38 us, with
// three stages one after the other 43).
constexpr int kWideK = 64;                // k per stage

// 16 (4) bytes per lane from a 64-bit address to LDS byte lds + 16 (4) *
// lane. The addresses are VGPRs: a buffer resource per copy piece would
// need more SGPRs than there are. The s_nop is the wait state between a
// write of M0 and its use here. live: all ones, or zero for a copy that
// counts as issued (vmcnt) but moves nothing; the wavefront's lanes are all
// active here.
__device__ __forceinline__ void dma16_g(const char *p, uint32_t lds, int live) {
    lds = __builtin_amdgcn_readfirstlane(lds);
    live = __builtin_amdgcn_readfirstlane(live);
    asm volatile("s_mov_b32 exec_lo, %2\n\ts_mov_b32 exec_hi, %2\n\t"
                 "global_load_lds_dwordx4 %0, off\n\ts_mov_b64 exec, -1"
                 ::"v"(p), "{m0}"(lds), "s"(live) : "memory");
}
__device__ __forceinline__ void dma4_g(const char *p, uint32_t lds) {
    lds = __builtin_amdgcn_readfirstlane(lds);
    asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(p), "{m0}"(lds) : "memory");
}

// Tile (o0, m0) of 64 TO outputs x 64 TMM rows. sw workgroups of this XCD
// share its w rows (this one is number iw of them), 32 / sw its x rows
// (number ix). A stage in LDS: BO w rows, then BM x rows, of 128 bytes;
// 16-byte chunk c of row r at slot c ^ (r % 8), so that the 8 rows of one
// LDS read phase hit 8 distinct slots. K is a multiple of 32: an odd last
// half stage has no second half to read, so its copies repeat the first.
template <int TO, int TMM, int ST>
__device__ __forceinline__ void gemm_wide(char *sm, const GemmSegs &sg, const uint16_t *x, int M,
                                          int K, int o0, int m0, int sw, int iw, int ix) {
    constexpr int NW = 4, BO = 64 * TO, BM = 64 * TMM;
    constexpr int PB = BO * 128, SB = (BO + BM) * 128;
    constexpr int PPW = (BO + BM) / 8 / NW, NF = TO * TMM, NR = TO + TMM;
    static_assert((BO + BM) / 8 % NW == 0, "copy pieces must split evenly over the wavefronts");
    const int O = sg.row0[sg.n];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wo = wave >> 1, wm = wave & 1;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_void *)sm);
    const int nk = (K + kWideK - 1) / kWideK;
    const bool odd = K % kWideK != 0;
    // this wavefront's copy pieces: 8 rows of 128 bytes each, in one
    // segment. Rows past O or M read the last row (their products are not
    // stored).
    const char *src[PPW];
    const int cg = (lane & 7) ^ (lane >> 3);               // chunk: slot ^ row % 8
    // the last stage's step back to its first half
    const int tail = odd && cg >= 4 ? -64 : 0;
#pragma unroll
    for (int i = 0; i < PPW; i++) {
        const int p = wave * PPW + i;
        const bool pw = p < BO / 8;
        const int ob = min(o0 + p * 8, O - 1), si = __builtin_amdgcn_readfirstlane(seg_of(sg, ob));
        const uint16_t *base = pw ? sg.w[si] : x;
        const int r = p * 8 + (lane >> 3);
        const int row = pw ? min(o0 + r, O - 1) - sg.row0[si] : min(m0 + r - BO, M - 1);
        src[i] = (const char *)(base + (size_t)row * K) + cg * 16 + (nk == 1 ? tail : 0);
    }
    const uint32_t piece0 = lds0 + wave * PPW * 1024;
    // copy i of the stage in flight into ring slot `slot`; its address then
    // moves on by adv, to the next stage
    auto copy = [&](int i, uint32_t slot, int adv, int live) {
        dma16_g(src[i], piece0 + slot + i * 1024, live);
        src[i] += adv;
    };
    // from stage st to st + 1 (past the last stage it stays)
    auto advance = [&](int st) { return st + 1 < nk ? 128 + (st + 2 == nk ? tail : 0) : 0; };
    // Prefetch into L2: this workgroup's share of the lines of its operand
    // tiles, one 4-byte load per line into an LDS row that nothing reads.
    // Every lane loads, so that the wait counts are the same in every
    // wavefront.
    const char *pf;
    {
        const int nw = (BO + sw - 1) / sw, sx = 32 / sw, nx = (BM + sx - 1) / sx;
        const int e = threadIdx.x;
        const bool px = e >= nw && e < nw + nx;
        const int o = min(o0 + iw * nw + (e < nw ? e : 0), O - 1), si = seg_of(sg, o);
        const int row = px ? min(m0 + ix * nx + e - nw, M - 1) : o - sg.row0[si];
        pf = (const char *)((px ? x : sg.w[si]) + (size_t)row * K) + min(ST, nk - 1) * 128;
    }
    auto prefetch = [&](int st) {            // stages ST, ST + 1, ... in turn
        dma4_g(pf, lds0 + ST * SB + wave * 256);
        pf += st + 1 < nk ? 128 : 0;
    };
    f32x16 acc[TO][TMM];
#pragma unroll
    for (int t = 0; t < TO; t++)
#pragma unroll
        for (int u = 0; u < TMM; u++) acc[t][u] = f32x16{};
    struct Frag {
        bf16x8 a[TO], b[TMM];
    };
    // chunk 2 s + lane / 32 of row lane % 32 of a 32-row block, s = 0
    const uint32_t rbase = (lane & 31) * 128 + (((lane >> 5) ^ (lane & 7)) << 4);
    // operand read j of k16 step s of the stage in `slot`, in the order the
    // MFMAs use them: a[0], b[0..], a[1..]
    auto rd1 = [&](uint32_t slot, int s, int j, Frag &f) {
        const char *p = sm + ((rbase ^ (s << 5)) + slot);
        if (j == 0 || j > TMM) {
            const int t = j == 0 ? 0 : j - TMM;
            f.a[t] = *reinterpret_cast<const bf16x8 *>(p + wo * TO * 4096 + t * 4096);
        } else {
            f.b[j - 1] = *reinterpret_cast<const bf16x8 *>(p + PB + wm * TMM * 4096 + (j - 1) * 4096);
        }
    };
    using no = std::false_type;
    using yes = std::true_type;
    // One k16 step: its NF MFMAs on f and, fenced in place between them, the
    // reads of the next step's operands into g (READ: k16 step s2 of slot
    // rslot) and the copies of a stage into cslot (COPY).
    auto step = [&](const Frag &f, Frag &g, auto read, uint32_t rslot, int s2, auto cpy,
                    uint32_t cslot, int adv, int live) {
        constexpr bool READ = decltype(read)::value, COPY = decltype(cpy)::value;
        int r = 0, d = 0;
#pragma unroll
        for (int i = 0; i < NF; i++) {
            acc[i / TMM][i % TMM] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                f.a[i / TMM], f.b[i % TMM], acc[i / TMM][i % TMM], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            // the reads go under the first three quarters of the MFMAs
#pragma unroll
            for (; READ && r < NR && (i == NF - 1 || r * NF * 3 <= i * NR * 4); r++) rd1(rslot, s2, r, g);
#pragma unroll
            for (; COPY && d < PPW && d * NF < (i + 1) * PPW; d++) copy(d, cslot, adv, live);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    Frag f0, f1;
    // stages 0 .. ST - 1 in flight; stage 0 published
#pragma unroll
    for (int st = 0; st < ST; st++) {
        const int adv = advance(st);
#pragma unroll
        for (int i = 0; i < PPW; i++) copy(i, st * SB, adv, (st - nk) >> 31);
    }
    prefetch(ST);
    // (the counts take every copy after the awaited ones as a live one)
    if (nk >= ST) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PPW * (ST - 1) + 1) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NR; j++) rd1(0, 0, j, f0);
    uint32_t slot = 0;
    for (int kt = 0; kt < nk - 1; kt++) {
        step(f0, f1, yes{}, slot, 1, no{}, 0, 0, 0);
        step(f1, f0, yes{}, slot, 2, no{}, 0, 0, 0);
        step(f0, f1, yes{}, slot, 3, no{}, 0, 0, 0);
        // every operand of this stage has been read, by this wavefront (it
        // waited for f1) and after the barrier by all, and the next stage has
        // landed (its copies are older than those of ST - 2 stages and the
        // last prefetch): stage kt + ST goes into this stage's slot
        if (kt + ST <= nk) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PPW * (ST - 2) + 1) : "memory");
        else asm volatile("s_waitcnt vmcnt(1)" ::: "memory");
        __syncthreads();
        const uint32_t next = slot + SB == ST * SB ? 0 : slot + SB;
        step(f1, f0, yes{}, next, 0, yes{}, slot, advance(kt + ST), (kt + ST - nk) >> 31);
        prefetch(kt + ST + 1);
        slot = next;
    }
    // the last stage; an odd K's second half is zeros
    auto mask = [&](Frag &f) {
        if (!odd) return;
#pragma unroll
        for (int t = 0; t < TO; t++) f.a[t] = bf16x8{};
#pragma unroll
        for (int u = 0; u < TMM; u++) f.b[u] = bf16x8{};
    };
    step(f0, f1, yes{}, slot, 1, no{}, 0, 0, 0);
    step(f1, f0, yes{}, slot, 2, no{}, 0, 0, 0);
    mask(f0);
    step(f0, f1, yes{}, slot, 3, no{}, 0, 0, 0);
    mask(f1);
    step(f1, f0, no{}, 0, 0, no{}, 0, 0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();                     // the ring is free: no copy in flight, no reader
    // Epilogue: lane -> m = lane % 32, o = 8 (i / 4) + 4 (lane / 32) + i % 4
    // of each 32 x 32 tile. Through LDS (this wavefront's quarter, rows m of
    // 64 TO bytes, 16-byte chunk c at c ^ (m % NCH)) so that the stores are
    // 16-byte pieces of whole rows; a row stored straight from the
    // accumulators would be 8-byte pieces of 32 rows per instruction.
    const int ow = o0 + wo * TO * 32, mw = m0 + wm * TMM * 32;
    bool vec = true;
    for (int i = 0; i < sg.n; i++)
        vec = vec && ((sg.ldy[i] | sg.row0[i] | sg.row0[i + 1]) & 7) == 0 && ((uintptr_t)sg.y[i] & 15) == 0;
    if (!vec) {
        store_tiles<TO, TMM>(sg, acc, ow, mw, O, M, lane);
        return;
    }
    constexpr int NCH = 4 * TO, ROW = 64 * TO;           // chunks, bytes of a row
    char *ep = sm + wave * (TMM * 32 * ROW);
#pragma unroll
    for (int t = 0; t < TO; t++)
#pragma unroll
        for (int u = 0; u < TMM; u++) {
            const int m = u * 32 + (lane & 31);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const f32x16 &v = acc[t][u];
                *reinterpret_cast<uint2 *>(ep + m * ROW + (((t * 4 + q) ^ (m & (NCH - 1))) << 4) +
                                           ((lane >> 5) << 3)) =
                    make_uint2(pk2(v[4 * q], v[4 * q + 1]), pk2(v[4 * q + 2], v[4 * q + 3]));
            }
        }
    // (own quarter only: a wavefront's LDS accesses execute in order)
    constexpr int RPI = 64 / NCH;                        // rows per instruction
    const int pc = lane & (NCH - 1);
    const int o = ow + pc * 8, si = seg_of(sg, min(o, O - 1));
    uint16_t *yo = sg.y[si] + (o - sg.row0[si]);
    const int ld = sg.ldy[si];
#pragma unroll 8
    for (int i = 0; i < TMM * 32 / RPI; i++) {
        const int m = i * RPI + lane / NCH;
        const uint4 v = *reinterpret_cast<const uint4 *>(ep + m * ROW + ((pc ^ (m & (NCH - 1))) << 4));
        if (o < O && mw + m < M) *reinterpret_cast<uint4 *>(yo + (size_t)(mw + m) * ld) = v;
    }
}

// A last output tile of at most 64 outputs (the GDN in-projection's gate
// rows: 12352 = 48 * 256 + 64) runs as a 64-wide tile, ids after the
// full tiles', instead of as a whole round of mostly empty 256-wide ones.
template <int TO>
__host__ __device__ inline bool wide_narrow(int O) { return TO == 4 && O % 256 > 0 && O % 256 <= 64 && O > 256; }

template <int TO, int TMM, int ST>
__global__ __launch_bounds__(256, TO * TMM <= 8 && ST == 2 ? 2 : 1) void k_gemm_wide(
    GemmSegs sg, const uint16_t *__restrict__ x, int M, int K) {
    constexpr int BO = 64 * TO, BM = 64 * TMM;
    __shared__ __attribute__((aligned(16))) char sm[ST * (BO + BM) * 128 + 1024];
    const int O = sg.row0[sg.n];
    const bool narrow = wide_narrow<TO>(O);
    const int nbo = narrow ? O / BO : (O + BO - 1) / BO, nbm = (M + BM - 1) / BM;
    const int n = tile_grid(nbo, nbm);
    // the workgroups of this one's XCD that share its tiles (tile_of)
    const int sw = min(nbm, 8);
    if (TO == 4 && (int)blockIdx.x >= n) {
        gemm_wide<1, TMM, ST>(sm, sg, x, M, K, nbo * BO, ((int)blockIdx.x - n) * BM, 1, 0, 0);
        return;
    }
    int ob, mb;
    tile_of(blockIdx.x, nbo, nbm, ob, mb);
    if (ob >= nbo) return;                      // (the grid is a multiple of 8)
    gemm_wide<TO, TMM, ST>(sm, sg, x, M, K, ob * BO, mb * BM, sw, mb % sw, ob % (32 / sw));
}

// y = rnd(sum over the splits of part, in split order), scattered to the
// segments; a thread owns 4 consecutive outputs of one row (O % 4 == 0)
__global__ __launch_bounds__(256) void k_gemm_reduce(GemmSegs sg, const float *__restrict__ part,
                                                     int M, int nsplit) {
    const int O = sg.row0[sg.n], O4 = O / 4;
    const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= (size_t)M * O4) return;
    const int m = (int)(e / O4), o = (int)(e % O4) * 4;
    float4 sm = *reinterpret_cast<const float4 *>(part + (size_t)m * O + o);
    for (int s = 1; s < nsplit; s++) {
        const float4 v = *reinterpret_cast<const float4 *>(part + ((size_t)s * M + m) * O + o);
        sm.x += v.x; sm.y += v.y; sm.z += v.z; sm.w += v.w;
    }
    const int si = seg_of(sg, o);
    uint16_t *yr = sg.y[si] + (size_t)m * sg.ldy[si] + (o - sg.row0[si]);
    yr[0] = f2bf(sm.x);
    yr[1] = f2bf(sm.y);
    yr[2] = f2bf(sm.z);
    yr[3] = f2bf(sm.w);
}

// timing / error names by GemmPlace
const char *const kTileNames[] = {"k_gemm_tile", "k_gemm_tile_in", "k_gemm_tile_out"};
const char *const kWideNames[] = {"k_gemm_wide", "k_gemm_wide_in", "k_gemm_wide_out"};

template <int WO, int WM, int TO, int TMM, int ST = kTileStages>
int launch_tile(const GemmSegs &sg, const uint16_t *x, int M, int K, GemmPlace place,
                int nsplit) {
    const char *name = kTileNames[place];
    constexpr int BO = 32 * TO * WO, BM = 32 * TMM * WM;
    const int O = sg.row0[sg.n];
    const int nbo = (O + BO - 1) / BO, nbm = (M + BM - 1) / BM;
    const unsigned grid = (unsigned)tile_grid(nbo, nbm);
    float *part = nullptr;
    if (nsplit > 1) {
        part = (float *)scratch(kScratchWork3, (size_t)nsplit * M * O * 4);
        if (!part) return kErrHip;
    }
    APUS_TIMED(name, k_gemm_tile<WO, WM, TO, TMM, ST><<<grid * nsplit, 64 * WO * WM, 0, stream()>>>(
                         sg, x, M, K, part, nsplit));
    if (int r = launch_check(name)) return r;
    if (nsplit > 1) {
        APUS_TIMED("k_gemm_reduce", k_gemm_reduce<<<cdiv((size_t)M * O / 4, 256), 256, 0,
                                                    stream()>>>(sg, part, M, nsplit));
        return launch_check("k_gemm_reduce");
    }
    return kOk;
}

template <int TO, int TMM, int ST>
int launch_wide(const GemmSegs &sg, const uint16_t *x, int M, int K, GemmPlace place) {
    const char *name = kWideNames[place];
    constexpr int BO = 64 * TO, BM = 64 * TMM;
    const int O = sg.row0[sg.n], nbm = (M + BM - 1) / BM;
    const bool narrow = wide_narrow<TO>(O);
    const unsigned grid = (unsigned)(tile_grid(narrow ? O / BO : (O + BO - 1) / BO, nbm) + (narrow ? nbm : 0));
    APUS_TIMED(name, k_gemm_wide<TO, TMM, ST><<<grid, 256, 0, stream()>>>(sg, x, M, K));
    return launch_check(name);
}

// Tile shapes and what they take, in us for K = 2048 (it scales with K for
// all of them), measured over 512 .. 12352 outputs x 16 .. 4096 rows: with
// up to one workgroup per CU `one`, of which `fill` only when all CUs have
// one (shared bandwidth); with two, `two` (the small shapes run 2 to 5
// workgroups per CU side by side). Small shapes win while they leave no CU
// with a second one, since a workgroup walks K alone; large ones move
// fewer operand bytes per product.
struct TileShape {
    int bo, bm;
    float one, fill, two;
    bool split;                             // has a K-split form
    int (*run)(const GemmSegs &, const uint16_t *, int, int, GemmPlace, int);
};
template <int TO, int TMM, int ST>
int run_wide(const GemmSegs &sg, const uint16_t *x, int M, int K, GemmPlace place, int) {
    return launch_wide<TO, TMM, ST>(sg, x, M, K, place);
}
const TileShape kTileShapes[] = {
    {64, 64, 12.7f, 0.0f, 20.5f, true, launch_tile<2, 1, 1, 2>},
    {128, 64, 15.5f, 0.0f, 33.0f, true, launch_tile<2, 2, 2, 1>},
    {128, 128, 24.0f, 6.5f, 50.0f, true, launch_tile<2, 4, 2, 1>},
    {128, 128, 27.0f, 2.0f, 41.5f, false, run_wide<2, 2, 2>},
    {128, 128, 22.5f, 3.0f, 47.0f, false, run_wide<2, 2, 3>},
    {128, 192, 27.5f, 3.0f, 62.0f, false, run_wide<2, 3, 3>},
    {256, 192, 49.0f, 10.0f, 97.0f, false, run_wide<4, 3, 2>},
    {256, 256, 62.0f, 12.0f, 124.0f, false, run_wide<4, 4, 2>},
};

}  // namespace

namespace apus {

// The shape with the least estimated time. Decode-sized row counts with a
// long K (the output projections, K = 4096) split K in two: twice the
// workgroups for the few output tiles (w_out at 325 rows: 27 -> 21 us). The
// split depends on M, K and whether the launch's outputs are a multiple of 4,
// and every shape accumulates an element's k16 steps in order, so a product's
// result is the same whichever shape computes it, and segmented or not where
// the launches agree on that.
int gemm_tile(const GemmSegs &sg, const uint16_t *x, size_t M, size_t K, GemmPlace place) {
    const int O = sg.row0[sg.n], cus = cu_count();
    const int nsplit = M <= 512 && K >= 4096 && O % 4 == 0 ? 2 : 1;
    const TileShape *best = nullptr;
    float tbest = 0.0f;
    for (const TileShape &t : kTileShapes) {
        if (nsplit > 1 && !t.split) continue;
        const bool narrow = t.bo == 256 && wide_narrow<4>(O);
        const size_t nbo = narrow ? O / t.bo : cdiv(O, t.bo);
        const size_t wgs = nbo * cdiv(M, t.bm) * nsplit;
        const int n = (int)((wgs + cus - 1) / cus);           // the busiest CU's
        const float last = (float)((wgs - 1) % cus + 1) / cus;  // CUs with that many
        const float us = (float)(n / 2) * t.two + (float)(n % 2) * t.one - t.fill * (1.0f - last) +
                         (narrow ? 10.0f : 0.0f);
        if (!best || us < tbest) {
            best = &t;
            tbest = us;
        }
    }
    return best->run(sg, x, (int)M, (int)K, place, nsplit);
}

// checks shared by the MFMA entry points: K a multiple of 32 (stages),
// 16-byte aligned operands (16-byte copies), byte offsets under 2 GiB
int gemm_tile_check(const uint16_t *x, size_t M, size_t O, size_t K) {
    if (int r = check_dims(M, O, K)) return r;
    if (!x) return set_error(kErrArgument, "NULL operand");
    if (K == 0 || K % 32 != 0 || (uintptr_t)x % 16 != 0)
        return set_error(kErrUnsupported, "MFMA gemm needs K a multiple of 32 and 16-byte "
                         "aligned operands (K=%zu)", K);
    if (O * K * 2 >= 0x7fff0000u || M * K * 2 >= 0x7fff0000u)
        return set_error(kErrUnsupported, "MFMA gemm operands must stay under 2 GiB");
    return kOk;
}

int launch_seq(const uint16_t *w, const uint16_t *x, uint16_t *y, size_t M, size_t O,
               size_t K) {
    if (int r = check_dims(M, O, K)) return r;
    if (M == 0 || O == 0) return kOk;
    if (M > 65535) return set_error(kErrUnsupported, "sequential gemm takes up to 65535 rows");
    // (K = 0, zeros, has no pieces to load ahead and no rows per workgroup
    // below: the scalar kernel, which reads nothing then)
    const bool vec = K != 0 && K % 8 == 0 && ((uintptr_t)w | (uintptr_t)x) % 16 == 0;
    const dim3 grid(cdiv(O, 64), (unsigned)M);
    if (vec) {
        if (K * 2 > 64 * 1024) return set_error(kErrUnsupported, "sequential gemm takes K up to 32768");
        // rows per workgroup: no more than give every CU one (a chain that
        // shares its SIMD with another is slower: 4 x 8192 x 2048 20.0 us with
        // four, 16.8 with two), x rows as fp32 in at most 64 KiB of LDS
        const int R = (int)std::min<size_t>({M, 4, 16384 / K, cdiv(cdiv(O, 64) * M, cu_count())});
        if (K % kSeqK == 0 && R > 0)
            APUS_TIMED("k_gemm_seq64",
                       k_gemm_seq64<<<dim3(grid.x, cdiv(M, R)), 64 * (4 + R), R * K * 4, stream()>>>(
                           w, x, y, (int)M, (int)O, (int)K, R));
        else if (K * 4 <= 64 * 1024)
            APUS_TIMED("k_gemm_seq",
                       k_gemm_seq<true, true><<<grid, 64, K * 4, stream()>>>(w, x, y, (int)O, (int)K));
        else
            APUS_TIMED("k_gemm_seq",
                       k_gemm_seq<true><<<grid, 64, K * 2, stream()>>>(w, x, y, (int)O, (int)K));
    } else {
        APUS_TIMED("k_gemm_seq", k_gemm_seq<false><<<grid, 64, 0, stream()>>>(w, x, y, (int)O, (int)K));
    }
    return launch_check("k_gemm_seq");
}

// Device copies of host weights, keyed by host address (and size).
struct WeightCopy {
    void *dev = nullptr;
    size_t bytes = 0;
    int device = -1;
};
std::unordered_map<const void *, WeightCopy> g_weights;

const uint16_t *weight_copy(const uint16_t *w, size_t bytes) {
    WeightCopy &e = g_weights[w];
    const int dev = current_device();
    if (e.dev && (e.bytes != bytes || e.device != dev)) {
        if (e.device == dev) (void)hipFree(e.dev);
        e = WeightCopy{};
    }
    if (!e.dev) {
        if (hipMalloc(&e.dev, bytes) != hipSuccess) {
            e = WeightCopy{};
            set_error(kErrHip, "weight copy: hipMalloc of %zu bytes failed", bytes);
            return nullptr;
        }
        if (hipMemcpyAsync(e.dev, w, bytes, hipMemcpyHostToDevice, stream()) != hipSuccess) {
            set_error(kErrHip, "weight copy: upload of %zu bytes failed", bytes);
            return nullptr;
        }
        e.bytes = bytes;
        e.device = dev;
    }
    return (const uint16_t *)e.dev;
}

int host_gemm(const uint16_t *w, const uint16_t *x, uint16_t *y, size_t M, size_t O, size_t K) {
    APUS_READY();
    if (int r = check_dims(M, O, K)) return r;
    if (M == 0 || O == 0) return kOk;
    if (!w || !x || !y) return set_error(kErrArgument, "NULL operand");
    const uint16_t *dw = weight_copy(w, O * K * 2);
    if (!dw && O * K) return kErrHip;
    APUS_STAGE(dx, uint16_t, kScratchIn, x, M * K * 2);
    uint16_t *dy = (uint16_t *)scratch(kScratchOut, M * O * 2);
    if (!dy) return kErrHip;
    if (int r = launch_seq(dw, dx, dy, M, O, K)) return r;
    return stage_out(y, dy, M * O * 2);
}

}  // namespace apus

extern "C" {

int apus_hip_bf16_gemv(const uint16_t *w, const uint16_t *x, uint16_t *y, size_t O, size_t K) {
    return host_gemm(w, x, y, 1, O, K);
}

int apus_hip_bf16_gemm(const uint16_t *w, const uint16_t *x, uint16_t *y, size_t M, size_t O,
                       size_t K) {
    return host_gemm(w, x, y, M, O, K);
}

int apus_hip_bf16_weights_release(void) {
    APUS_READY();
    APUS_HIP_TRY(hipStreamSynchronize(stream()));
    const int dev = current_device();
    for (auto &kv : g_weights)
        if (kv.second.dev && kv.second.device == dev) (void)hipFree(kv.second.dev);
    g_weights.clear();
    return kOk;
}

int apus_hip_bf16_gemm_dev(const uint16_t *w, const uint16_t *x, uint16_t *y, size_t M,
                           size_t O, size_t K) {
    APUS_READY();
    return launch_seq(w, x, y, M, O, K);
}

int apus_hip_bf16_gemm_mfma_dev(const uint16_t *w, const uint16_t *x, uint16_t *y, size_t M,
                                size_t O, size_t K) {
    APUS_READY();
    if (M == 0 || O == 0) return check_dims(M, O, K);
    if (!w || !y) return set_error(kErrArgument, "NULL operand");
    if (int r = gemm_tile_check(x, M, O, K)) return r;
    if ((uintptr_t)w % 16 != 0)
        return set_error(kErrUnsupported, "MFMA gemm needs 16-byte aligned operands");
    GemmSegs sg{};
    sg.n = 1;
    sg.row0[1] = (int)O;
    sg.w[0] = w;
    sg.y[0] = y;
    sg.ldy[0] = (int)O;
    return gemm_tile(sg, x, M, K, kGemmAlone);
}

}  // extern "C"
