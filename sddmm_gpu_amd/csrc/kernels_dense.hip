// Dense-block kernel of the SDDMM engine for gfx950 (MI355X).
//
// Where S has a dense core (heavy rows x popular columns of a power-law
// matrix), the sampled products of a 128 x 128 block are cheaper as one dense
// contraction on the matrix cores than as gathered dot products on the
// vector ALU: a block of 128 rows (any rows, given by a list) times 128 columns
// (any columns, given by a list) is computed whole, left in LDS, and the block's
// nonzeros pick their entries from there, scale them by S.val and store them at
// their own positions of the output.  Structural zeros of the block are computed
// and dropped; the planner only hands over blocks dense enough for that to pay.
//
// Arithmetic.  The fp32 matrix instruction runs at a sixteenth of the bf16 one, so
// every operand is cut into three bf16 parts whose sum it is exactly (8 + 8 + 8
// significant bits), and eight of the nine products of parts are taken; the one left
// out, of the two last parts, is at most 2^-34 of the product.  A part is at most 2^-8
// of the one before it, so two of the others reach 2^-25 of the product: leaving them
// out as well would show where a sum has few products.  The matrix instruction does
// not round its sums to nearest either (a product alone comes out up to 2^-23 off), so
// it adds up 16 elements of K at a time, the products of the first parts (exact for
// one alone) apart from the seven small ones, and vector instructions, which round to
// nearest, add the two to the running sum.  Error against 64 bits over the blocks
// of a recommender matrix (relative, 2-norm; fp32 matrix instruction -> parts):
// K = 128 1.72e-7 -> 0.73e-7, K = 512 3.32e-7 -> 1.06e-7, all-positive factors at 512
// 2.83e-7 -> 0.77e-7, factors spread over e^(+-9) 9.2e-8 -> 7.2e-8; a product alone in
// its row 2.53e-8 -> 2.53e-8 (at most 2^-24 (1 + 2^-7) of it), four in a row 4.6e-8 ->
// 4.9e-8 (4.8e-8 for the chain of fp32 FMAs of the other kernels).  (Six products summed
// into one accumulator, 0.70 ms where this takes 0.84: 2.8e-7 at K = 512, but 3.2e-8 and up
// to 2.4 x 2^-24 for a product alone, 7.3e-8 for four.)  What parts cannot
// carry -- infinities, NaNs, sums beyond the range, values with bits under bf16's
// smallest subnormal -- is found and those results are computed once more in fp32
// (redo_picks).
//
// One workgroup of 4 waves per block, each wave a 64 x 64 quarter (2 x 2 MFMA
// tiles of 32 x 32, 64 accumulator registers).  K runs in chunks of 32: the
// chunk's 128 x 32 slices of the W rows and of the H rows are gathered from
// global memory into registers while the previous chunk is multiplied, cut into
// their parts among its last 32 matrix instructions, and written to LDS.  One
// buffer: two would leave room for one workgroup per CU only, and the second workgroup
// is what works while the first passes its barriers.  What bounds it is the matrix
// cores and the vector ALU about alike: per chunk and wave 2048 clocks of matrix
// instructions, 1800 of cutting and adding, and per workgroup 1150 of LDS reads and
// writes, two workgroups on a CU.  A tile's sums are added among the products of the
// tile after it (0.88 -> 0.84 ms; all four tiles' sums at a time do not fit the
// registers).  Recommender shape, 59.4 M nonzeros, K = 512: 1.03 ms with the fp32
// instruction, 0.84 with parts; K = 384 0.80 and 0.66 (8 x 95 GFLOP take 0.3 ms at the
// nominal bf16 rate; picking and storing 14 B per nonzero about 0.2).
#include <hip/hip_runtime.h>
#include <type_traits>
#include "kernels.hpp"
#include "bf16_parts.hpp"

using namespace sddmm;

namespace {

constexpr int kT = kDenseTile;           // 128 rows and 128 columns per block
constexpr int kKC = 32;                  // K elements per chunk
constexpr int kPartB = kKC * 2;          // bytes of one part of a staged row
constexpr int kRowB = 3 * kPartB + 16;   // bytes per staged row: 13 times 16, odd, so 16 rows spread over all banks
constexpr int kStageB = kT * kRowB;      // bytes per staged operand
constexpr int kCRowF = kT + 8;           // floats per row of the result block in LDS
constexpr int kLdsB = 2 * kStageB > kT * kCRowF * 4 ? 2 * kStageB : kT * kCRowF * 4;

// Workgroup barrier that orders LDS traffic only.  __syncthreads() also waits for every global
// load and store in flight (its workgroup-scope fence), which would drain the requests this kernel
// keeps in the air across its barriers: the next chunk's operands, the block's nonzero list, the
// stores of the block before.  Global memory is never used for communication inside a workgroup here.
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

__global__ __launch_bounds__(256, 2)
void sddmm_dense_kernel(const DenseArgs a)
{
    __shared__ __attribute__((aligned(16))) unsigned char lds[kLdsB];  // A B | result block
    __shared__ uint32_t inexact;  // nonzero: some operand of the block has bits below its three parts
    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int wr = wave >> 1, wc = wave & 1;  // this wave's 64 x 64 quarter
    const int m = lane & 31, kh = lane >> 5;
    const uint32_t K4 = (uint32_t)(a.K >> 2);
    const int n_chunks = a.K / kKC;
    const vec4f *__restrict__ W4 = reinterpret_cast<const vec4f *>(a.W);
    const vec4f *__restrict__ H4 = reinterpret_cast<const vec4f *>(a.H);
    // staging: thread t carries float4 q and q + 4 of rows r0 and r0 + 64 of both operands.  They go
    // side by side into LDS; the order of the K elements is the same for both operands, so it does not matter.
    //  16 neighbouring lanes write four rows that lie 4 apart: 64 different banks.
    const int q = t & 3, r0 = 16 * wave + 4 * ((t >> 2) & 3) + ((t >> 4) & 3);

    // Workgroup b works on slots b, b + grid, ...; its filled slots come first.
    int slot = blockIdx.x;
    if (slot >= a.n_slots) return;
    int2 range = a.slot_range[slot];
    if (range.y <= range.x) return;

    // float4 index of this thread's first piece of each of its rows of W and H at chunk 0
    auto load_ids = [&](int s, uint32_t (&wofs)[2], uint32_t (&hofs)[2]) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            wofs[i] = (uint32_t)a.slot_rows[s * kT + r0 + 64 * i] * K4 + (uint32_t)q;
            hofs[i] = (uint32_t)a.slot_cols[s * kT + r0 + 64 * i] * K4 + (uint32_t)q;
        }
    };
    vec4f ga[4], gb[4];
    auto fetch = [&](const uint32_t (&wofs)[2], const uint32_t (&hofs)[2]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) ga[i] = W4[wofs[i >> 1] + 4 * (i & 1)];
#pragma unroll
        for (int i = 0; i < 4; ++i) gb[i] = H4[hofs[i >> 1] + 4 * (i & 1)];
    };
    uint32_t lost = 0;  // of the operands staged by this thread for the block in hand
    vec4w pa[2][3], pb[2][3];
    auto split_part = [&](int k) {  // a quarter of it
        const int i = k >> 1;
        if (k & 1) split8(gb[2 * i], gb[2 * i + 1], pb[i], lost);
        else split8(ga[2 * i], ga[2 * i + 1], pa[i], lost);
    };
    auto split = [&]() {
#pragma unroll
        for (int k = 0; k < 4; ++k) split_part(k);
    };
    auto stage = [&]() {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                unsigned char *at = lds + (r0 + 64 * i) * kRowB + p * kPartB + 16 * q;
                *reinterpret_cast<vec4w *>(at) = pa[i][p];
                *reinterpret_cast<vec4w *>(at + kStageB) = pb[i][p];
            }
    };
    // One round of the block's nonzero list: 8 entries per thread, strided by the workgroup.
    constexpr int U = 8;
    struct Round { int p[U]; uint32_t rc[U]; float v[U]; };
    auto load_round = [&](Round &r, int first, int n1) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int idx = min(first + 256 * u, n1 - 1);  // clamped: no load behind a branch
            r.p[u] = a.nz_p[idx];
            r.rc[u] = a.nz_rc[idx];
            r.v[u] = a.nz_val ? a.nz_val[idx] : 1.0f;
        }
    };
    const float *Cb = reinterpret_cast<const float *>(lds);
    // Picks that are not stored from the result block but once more computed in fp32: all of a block
    // whose operands three parts do not hold, and any that come out as an infinity or a NaN (there is
    // one among the operands, or a sum left the range).
    bool redo = false, left = false;
    auto redo_picks = [&](int first, int n1) {
        for (int idx = first; idx < n1; idx += 256) {
            const uint32_t rc = a.nz_rc[idx];
            if (!redo && fabsf(Cb[(rc >> 8) * kCRowF + (rc & 255u)]) < INFINITY) continue;
            const vec4f *w = W4 + (uint32_t)a.slot_rows[slot * kT + (int)(rc >> 8)] * K4;
            const vec4f *h = H4 + (uint32_t)a.slot_cols[slot * kT + (int)(rc & 255u)] * K4;
            float d = 0.f;
#pragma unroll 1
            for (uint32_t k = 0; k < K4; ++k) {
                const vec4f x = w[k], y = h[k];
                d = fmaf(x.x, y.x, d); d = fmaf(x.y, y.y, d); d = fmaf(x.z, y.z, d); d = fmaf(x.w, y.w, d);
            }
            const int p = a.nz_p[idx];
            const float v = a.nz_val ? a.nz_val[idx] : a.val ? a.val[p] : 1.0f;
            a.out[p] = a.residual ? v - d : v * d;
        }
    };
    auto store_round = [&](Round &r, int first, int n1) {
        if (!a.nz_val && a.val) {
#pragma unroll
            for (int u = 0; u < U; ++u) r.v[u] = a.val[r.p[u]];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float dot = Cb[(r.rc[u] >> 8) * kCRowF + (r.rc[u] & 255u)];
            const bool keep = !redo && fabsf(dot) < INFINITY;
            left |= !keep;
            if (keep && first + 256 * u < n1) a.out[r.p[u]] = a.residual ? r.v[u] - dot : r.v[u] * dot;
        }
    };

    uint32_t wofs[2], hofs[2];
    load_ids(slot, wofs, hofs);
    fetch(wofs, hofs);
    if (t == 0) inexact = 0;
    split();
    stage();
    lds_barrier();
    for (;;) {
        // what the next block needs is requested while this one is computed: its row and column
        // lists now, the first chunk of its operands during this block's last chunk
        const int nslot = slot + (int)gridDim.x;
        int2 nrange = make_int2(0, 0);
        if (nslot < a.n_slots) nrange = a.slot_range[nslot];
        const bool has_next = nrange.y > nrange.x;
        uint32_t nw[2], nh[2];
        load_ids(has_next ? nslot : slot, nw, nh);

        floatx16 acc[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
        const unsigned char *ap = lds + (wr * 64 + m) * kRowB + kh * 16;
        const unsigned char *bp = lds + kStageB + (wc * 64 + m) * kRowB + kh * 16;
        // 16 elements of K, one 32 x 32 tile after the other, a tile's sums added to the running ones among the products
        // of the tile after it; between(k) is further vector work to be done among the products of tile k
        const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        floatx16 low = zero, high = zero;
        auto add = [&](int k) {
            floatx16 &sum = acc[k >> 1][k & 1];
            sum += high + low;
            asm volatile("" : "+v"(sum));  // (added here: left alone the compiler sinks it to where the sums are read)
        };
        auto products = [&](auto step, auto between) {
            constexpr int s = decltype(step)::value;
            bf16x8 av[2][3], bv[2][3];
#pragma unroll
            for (int p = 2; p >= 0; --p)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    av[i][2 - p] = *reinterpret_cast<const bf16x8 *>(ap + 32 * i * kRowB + (2 - p) * kPartB + 32 * s);
                    bv[i][p] = *reinterpret_cast<const bf16x8 *>(bp + 32 * i * kRowB + p * kPartB + 32 * s);
                }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = k >> 1, j = k & 1;
                constexpr int pp[7] = {1, 2, 0, 1, 2, 0, 1}, qq[7] = {2, 1, 2, 1, 0, 1, 0};
                floatx16 l = zero;  // small ones first
#pragma unroll
                for (int pq = 0; pq < 7; ++pq) l = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[i][pp[pq]], bv[j][qq[pq]], l, 0, 0, 0);
                if (s + k > 0) add((k + 3) & 3);
                const floatx16 h = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[i][0], bv[j][0], zero, 0, 0, 0);
                between(k);
                low = l;
                high = h;
                __builtin_amdgcn_sched_barrier(0);
            }
            if (s == 1) add(3);
        };
        for (int c = 0; c + 1 < n_chunks; ++c) {
            // the next chunk's loads are issued before this chunk's arithmetic, and what they bring is
            // cut into its parts between the chunk's later products
#pragma unroll
            for (int i = 0; i < 2; ++i) { wofs[i] += kKC / 4; hofs[i] += kKC / 4; }
            fetch(wofs, hofs);
            __builtin_amdgcn_sched_barrier(0);
            products(std::integral_constant<int, 0>{}, [](int) {});
            products(std::integral_constant<int, 1>{}, split_part);
            lds_barrier();  // everyone has read this chunk
            stage();
            lds_barrier();
        }
        fetch(nw, nh);  // the last chunk: the next block's first
        Round r0d;      // and the first round of this block's nonzero list
        load_round(r0d, range.x + t, range.y);
        __builtin_amdgcn_sched_barrier(0);
        products(std::integral_constant<int, 0>{}, [](int) {});
        products(std::integral_constant<int, 1>{}, [](int) {});
        if (lost & 0xffffu) inexact = 1;  // (read after the next barriers; any writer writes the same)
        lost = 0;
        lds_barrier();  // everyone has read the last chunk
        // the 128 x 128 block of dot products into LDS (over the staging buffers, which everyone has
        // left): register v of lane (m, kh) of tile (i, j) holds row 8*(v/4) + 4*kh + v%4, column m
        float *Cw = reinterpret_cast<float *>(lds);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int row = wr * 64 + i * 32 + 8 * (v >> 2) + 4 * kh + (v & 3);
                    const int col = wc * 64 + j * 32 + m;
                    Cw[row * kCRowF + col] = acc[i][j][v];
                }
        // The block's nonzeros pick their dot products, in rounds of 8 per thread: the first round is
        // here already, the next three are requested together before it is worked on (four rounds
        // cover a block that is half full; fuller ones take further steps of four rounds).
        {
            const int first = range.x + t, n1 = range.y;
            constexpr int R = 256 * U;
            Round r1d, r2d, r3d;
            load_round(r1d, first + R, n1);
            load_round(r2d, first + 2 * R, n1);
            load_round(r3d, first + 3 * R, n1);
            lds_barrier();
            redo = inexact != 0;
            left = false;
            store_round(r0d, first, n1);
            store_round(r1d, first + R, n1);
            store_round(r2d, first + 2 * R, n1);
            store_round(r3d, first + 3 * R, n1);
            for (int f = first + 4 * R; f < n1 + t; f += 4 * R) {  // (uniform bound: first - t + 4R.. < n1)
                load_round(r0d, f, n1);
                load_round(r1d, f + R, n1);
                load_round(r2d, f + 2 * R, n1);
                load_round(r3d, f + 3 * R, n1);
                store_round(r0d, f, n1);
                store_round(r1d, f + R, n1);
                store_round(r2d, f + 2 * R, n1);
                store_round(r3d, f + 3 * R, n1);
            }
            if (left) redo_picks(first, n1);
        }
        lds_barrier();  // the next block's staging overwrites the result block
        if (!has_next) break;
        split();  // the next block's first chunk has been in registers since this block's last chunk
        stage();
        if (t == 0) inexact = 0;
        lds_barrier();
        slot = nslot;
        range = nrange;
#pragma unroll
        for (int i = 0; i < 2; ++i) { wofs[i] = nw[i]; hofs[i] = nh[i]; }
    }
}

}  // namespace

namespace sddmm {

DenseFn dense_kernel() { return (DenseFn)sddmm_dense_kernel; }

}  // namespace sddmm
