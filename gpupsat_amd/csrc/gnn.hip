// gnn.hip -- the learned branching network: message passing over the literal-clause
// incidence graph, trained and run on the GPU (no reference counterpart).
//
// Nodes: 2n literal nodes and m clause nodes per instance, instances back to back;
// an edge per clause occurrence.  Hidden size 64, R rounds, weights shared by rounds:
//   H_l^0 = occ(l)/8 u_l + v_l                       H_c^0 = len(c)/4 u_c + v_c
//   M_c = 1/4 sum_{l in c} H_l     H_c' = relu([H_c | M_c] W_c^T + b_c)
//   M_l = 1/8 sum_{c ni l} H_c'    H_l' = relu([H_l | M_l | H_{not l}] W_l^T + b_l)
//   Z_v = [H_{2v+1} | H_{2v}]      R_v = relu(Z_v W_o^T + b_o)   Y_v = R_v W_y^T + b_y
// Y_v = (branching score, phase logit).  The three 64-wide products run on MFMA
// (v_mfma_f32_16x16x32_bf16): BF16 weights and BF16 inputs, FP32 accumulation.
// Aggregations, biases, the 2-output head, the loss and Adam are FP32.  Gradients and the
// loss are summed from per-workgroup partials in a fixed order, never
// with floating-point atomics, so they are reproducible bit for bit.
//
// Each half round is one kernel per direction (gather, product and elementwise work on rows
// held in registers), as memory traffic and its latency bound the network, not arithmetic: the 172
// GFLOP of a training pass over 512 x (n=300, m=1278) would take 0.15 ms at half of the MFMA
// peak, moving its rows of ~4.6 GB about 1 ms.  The pass takes 1.75 ms, where separate gather, product,
// mask and reduction kernels moved ~9 GB in 3.70 ms; a layer's kernel runs at 3-4.3 TB/s of
// compulsory bytes.
#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/gpsat.h"
#include "common.hpp"
#include "gpsat_internal.hpp"

namespace gpsat {
namespace gnn {

constexpr int HID = 64;
typedef uint16_t bf16_t;
typedef float f32x4 __attribute__((ext_vector_type(4)));

// parameter layout (FP32 master copy), in this order
constexpr int O_UL = 0, O_VL = 64, O_UC = 128, O_VC = 192;
constexpr int O_WC = 256, O_BC = O_WC + 64 * 128, O_WL = O_BC + 64, O_BL = O_WL + 64 * 192;
constexpr int O_WO = O_BL + 64, O_BO = O_WO + 64 * 128, O_WY = O_BO + 64, O_BY = O_WY + 2 * 64;
constexpr int N_PARAMS = O_BY + 2;

__device__ __forceinline__ bf16_t to_bf16(float f)
{
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (bf16_t)(u >> 16);
}
__device__ __forceinline__ float from_bf16(bf16_t h) { return __uint_as_float((uint32_t)h << 16); }

// ---------------------------------------------------------------------------------------
// Fragments.  v_mfma_f32_16x16x32_bf16 (gfx950) on a wave of 64: lane l supplies the 8
// consecutive-k values A[l%16][8(l/16) .. 8(l/16)+7] and B[8(l/16) .. 8(l/16)+7][l%16] and
// receives D[4(l/16)+j][l%16] (j = 0..3).  Every product is computed transposed, weights as
// A and node rows as B, so lane l = 16q + r works on row r of the wavefront's 16: of each 64
// columns it supplies the 16 columns in(i) = 32 (i/8) + 8q + i%8 and receives the 16 columns
// out(i) = 16 (i/4) + 4q + i%4, i = 0..15.  (The k index is in the order of the columns: with
// another order the FP32 sums round differently, and a BF16 rounding after them now and then.)
// Memory is read and written in another lane order with the same columns: lane 4r + q, so that
// four neighbouring lanes share a row and a float4 access of theirs falls in one 128-byte line
// (with the product's own lane order every lane of a quad is on another row, and the address
// unit takes four times as long: the clause layer took 168 us instead of 146).  Registers change
// order through ds_bpermute, rows in BF16 on the way in and results in FP32 on the way out
// (to_product, from_product).  So a layer is gather -> BF16 -> MFMA -> ReLU -> store without a
// trip through memory.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ bf16x8 ld8(const bf16_t* p) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p)); }
// (rows kept for the backward pass or the weight gradient: read again only after far more than
// a cache's worth of other rows, so stored past the caches; clause layer 146 -> 130 us, literal
// layer 123 -> 102 us at 654,336 clauses and 307,200 literals)
__device__ __forceinline__ void st8(bf16_t* p, bf16x8 v)
{
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    __builtin_nontemporal_store(__builtin_bit_cast(i32x4, v), reinterpret_cast<i32x4*>(p));
}
__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// 8 floats rounded to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ bf16x8 pack8(const float* x)
{
    bf16x8 v;
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = (__bf16)x[i];
    return v;
}
// this lane's 16 values of a 64-wide FP32 row: the columns in(i), or out(i).  NT: past the caches,
// for rows that are next touched after more than they hold.
typedef float v4f __attribute__((ext_vector_type(4)));
template <bool OUT = false, bool NT = false>
__device__ __forceinline__ void ld_row(float (&x)[16], const float* row, int q)
{
    const v4f* p = reinterpret_cast<const v4f*>(row) + (OUT ? q : 2 * q);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const v4f* a = p + (OUT ? 4 * k : 8 * (k >> 1) + (k & 1));
        const v4f v = NT ? __builtin_nontemporal_load(a) : *a;
#pragma unroll
        for (int j = 0; j < 4; j++) x[4 * k + j] = v[j];
    }
}
template <bool NT = false>
__device__ __forceinline__ void st_row(float* row, const float (&x)[16], int q)   // columns out(i)
{
    v4f* p = reinterpret_cast<v4f*>(row + 4 * q);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const v4f v = {x[4 * k], x[4 * k + 1], x[4 * k + 2], x[4 * k + 3]};
        if (NT) __builtin_nontemporal_store(v, p + 4 * k);
        else p[4 * k] = v;
    }
}
// the same values of the neighbouring row (l ^ 1: the other polarity of the variable)
__device__ __forceinline__ bf16x8 flip8(bf16x8 v)
{
    uint4 w = __builtin_bit_cast(uint4, v);   // (product lane order)
    w.x = __builtin_amdgcn_mov_dpp(w.x, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
    w.y = __builtin_amdgcn_mov_dpp(w.y, 0xB1, 0xF, 0xF, false);
    w.z = __builtin_amdgcn_mov_dpp(w.z, 0xB1, 0xF, 0xF, false);
    w.w = __builtin_amdgcn_mov_dpp(w.w, 0xB1, 0xF, 0xF, false);
    return __builtin_bit_cast(bf16x8, w);
}
// between the lane orders of memory (4r + q) and of the products (16q + r)
__device__ __forceinline__ int lane_perm(int x, int from) { return __builtin_amdgcn_ds_bpermute(from, x); }
__device__ __forceinline__ bf16x8 to_product(bf16x8 v, int lane)
{
    const int from = 4 * (4 * (lane & 15) + (lane >> 4));
    const uint4 w = __builtin_bit_cast(uint4, v);
    return __builtin_bit_cast(bf16x8, uint4{(uint32_t)lane_perm(w.x, from), (uint32_t)lane_perm(w.y, from),
                                            (uint32_t)lane_perm(w.z, from), (uint32_t)lane_perm(w.w, from)});
}
__device__ __forceinline__ void from_product(float (&x)[16], int lane)
{
    const int from = 4 * (16 * (lane & 3) + (lane >> 2));
#pragma unroll
    for (int i = 0; i < 16; i++) x[i] = __int_as_float(lane_perm(__float_as_int(x[i]), from));
}
__device__ __forceinline__ float flip1(float x)
{
    return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0xB1, 0xF, 0xF, false));
}

// Weights [R x KW] (row-major BF16) into LDS, rows padded by 16 bytes (the 16 rows a wave
// reads at once fall in different banks).
template <int R, int KW>
__device__ __forceinline__ void stage_weights(bf16_t* s, const bf16_t* __restrict__ W)
{
    for (int i = threadIdx.x; i < R * KW / 8; i += blockDim.x) {
        const int c = (8 * i) / KW, k = (8 * i) % KW;
        *reinterpret_cast<uint4*>(s + c * (KW + 8) + k) = reinterpret_cast<const uint4*>(W)[i];
    }
}
// x[i] = the product's output column 64B + out(i): KS k-steps of 32 against the staged rows
// (f and x in product lane order)
template <int KS>
__device__ __forceinline__ void product(float (&x)[16], const bf16_t* s, int B, const bf16x8 (&f)[KS], int lane)
{
    constexpr int SK = 32 * KS + 8;
    int at = (64 * B + (lane & 15)) * SK + 8 * (lane >> 4);
    asm volatile("" : "+v"(at));   // weights stay in LDS: hoisted out of the tile loop they spill
#pragma unroll
    for (int ct = 0; ct < 4; ct++) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < KS; k++) acc = mfma32(ld8(s + at + 16 * ct * SK + 32 * k), f[k], acc);
#pragma unroll
        for (int j = 0; j < 4; j++) x[4 * ct + j] = acc[j];
    }
}

// value of lane J of the quad, in each of its four lanes
template <int J>
__device__ __forceinline__ int quad_lane(int x) { return __builtin_amdgcn_mov_dpp(x, 0x55 * J, 0xF, 0xF, false); }

__device__ __forceinline__ uint32_t quad_or(uint32_t x)
{
    x |= __builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, false);      // quad_perm [1,0,3,2]
    return x | __builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
}

// The edges of one row, read ahead: its offsets, and the index of its q-th neighbour of four in
// lane q (a load costs the address unit as much for one index in all four lanes as for four).
struct Edges {
    int e0, e1, id;
    __device__ __forceinline__ void offsets(const int32_t* __restrict__ off, int row, int q)
    {
        const int e = off[row + (q & 1)];
        e0 = quad_lane<0>(e);
        e1 = quad_lane<1>(e);
    }
    __device__ __forceinline__ void ids(const int32_t* __restrict__ edges, int e, int q)
    {
        id = edges[max(0, min(e + q, e1 - 1))];
    }
};
// s += sum over the row's edges of the neighbours' rows X[id], in edge order; two rows in
// flight, the next four edges' indices read meanwhile
__device__ __forceinline__ void gather_row(float (&s)[16], const int32_t* __restrict__ edges, Edges& E, int q,
                                           const float* __restrict__ X)
{
    auto add = [&](const float(&x)[16]) {
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] += x[i];
    };
    for (int e = E.e0; e < E.e1; e += 4) {
        const int k = E.e1 - e, v = E.id;
        float a[16], b[16];
        ld_row(a, X + (size_t)quad_lane<0>(v) * HID, q);
        if (k > 1) ld_row(b, X + (size_t)quad_lane<1>(v) * HID, q);
        if (k > 4) E.ids(edges, e + 4, q);
        add(a);
        if (k > 1) add(b);
        if (k > 2) {
            ld_row(a, X + (size_t)quad_lane<2>(v) * HID, q);
            if (k > 3) ld_row(b, X + (size_t)quad_lane<3>(v) * HID, q);
            add(a);
            if (k > 3) add(b);
        }
    }
}

// Workgroups go to the XCDs in turn (workgroup b to XCD b % 8): logical block of workgroup b
// such that each XCD takes one contiguous eighth of the rows, so an instance's rows stay in
// one XCD's L2 for the gathers of its neighbours.  The grid is a multiple of 8.
__device__ __forceinline__ int xcd_block() { return (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3); }

// x summed over the 16 rows, in every lane of its column quarter q: two rotations inside each
// 16 lanes, then the permlane swaps (no LDS); fixed order
__device__ __forceinline__ float row_sum(float x)
{
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x124, 0xF, 0xF, false));   // row_ror:4
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x128, 0xF, 0xF, false));   // row_ror:8
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_int(x), __float_as_int(x), false, false);
    x = __int_as_float(r[0]) + __int_as_float(r[1]);
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_int(x), __float_as_int(x), false, false);
    return __int_as_float(h[0]) + __int_as_float(h[1]);
}
// Workgroup totals of each wavefront's x[i] (column in(i) or out(i), over its rows) into
// out[64]; fixed order.  red: 64 floats a wavefront.
template <bool OUT>
__device__ __forceinline__ void block_sum(const float (&x)[16], float* red, float* out, int lane, int wave)
{
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const float v = row_sum(x[i]);
        if (lane < 4) red[64 * wave + (OUT ? 16 * (i >> 2) + 4 * lane + (i & 3) : 32 * (i >> 3) + 8 * lane + (i & 7))] = v;
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        float v = 0.f;
        for (int w = 0; w < (int)blockDim.x >> 6; w++) v += red[64 * w + threadIdx.x];
        out[threadIdx.x] = v;
    }
}

// Wavefronts of a layer's workgroup, which share the staged weights: 8 (instead of 4: the
// clauses' layer 132 -> 126 us, its backward 157 -> 142), but 4 where the first round's backward
// sums rows over the workgroup at several barriers (121 us; 8: 141).
constexpr int LAYER_WAVES = 8, LAST_WAVES = 4;

// One half round, whole: H' = relu([H | scale * sum of neighbours | (LIT) H of l ^ 1] W^T + b),
// 16 rows per wavefront, in place (a row is read and written by its own wavefront only, and the
// two rows of a variable share one).
//   FIRST  H is the embedding, computed from the degrees instead of read, the neighbours' too:
//          8 bytes of offsets per edge, looked up by the lane that holds its index, instead of a
//          256-byte row (added edge by edge in FP32 like any message: from the sum of the
//          occurrences it would be rounded differently)
//   TRAIN  X = bf16([H | messages]) and the sign mask of H' are kept for the backward pass
template <bool LIT, bool FIRST, bool TRAIN>
__global__ __launch_bounds__(64 * LAYER_WAVES, 4) void k_layer(const int32_t* __restrict__ off, const int32_t* __restrict__ edges,
                                                  const int32_t* __restrict__ n_off, int N, const float* __restrict__ th,
                                                  const bf16_t* __restrict__ W, const float* __restrict__ bias,
                                                  const float* __restrict__ Hn, float* H, bf16_t* __restrict__ X,
                                                  uint2* __restrict__ mask)
{
    constexpr int K = LIT ? 192 : 128, KS = K / 32;
    __shared__ __align__(16) bf16_t sW[64 * (K + 8)];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q = lane & 3;
    const int r = 16 * (xcd_block() * LAYER_WAVES + wave) + (lane >> 2), row = min(r, N - 1);
    Edges E;
    E.offsets(off, row, q);
    stage_weights<64, K>(sW, W);
    const int deg = E.e1 - E.e0;
    E.ids(edges, E.e0, q);
    float h[16], s[16], b[16];
    bf16x8 f[KS];
    if constexpr (FIRST) {
        ld_row(h, th + (LIT ? O_UL : O_UC), q);
        ld_row(b, th + (LIT ? O_VL : O_VC), q);
#pragma unroll
        for (int i = 0; i < 16; i++) h[i] = (float)deg * (LIT ? 0.125f : 0.25f) * h[i] + b[i];
    } else
        ld_row(h, H + (size_t)row * HID, q);
    if constexpr (FIRST && !LIT) {
        float u[16];
        ld_row(u, th + O_UL, q);
        ld_row(b, th + O_VL, q);
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = 0.f;
        auto add = [&](int occ) {
            const float w = (float)occ * 0.125f;
#pragma unroll
            for (int i = 0; i < 16; i++) s[i] += w * u[i] + b[i];
        };
        for (int e = E.e0; e < E.e1; e += 4) {
            const int k = E.e1 - e, occ = n_off[E.id + 1] - n_off[E.id];
            if (k > 4) E.ids(edges, e + 4, q);
            add(quad_lane<0>(occ));
            if (k > 1) add(quad_lane<1>(occ));
            if (k > 2) add(quad_lane<2>(occ));
            if (k > 3) add(quad_lane<3>(occ));
        }
    } else {
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = 0.f;
        gather_row(s, edges, E, q, Hn);
    }
#pragma unroll
    for (int i = 0; i < 16; i++) s[i] *= LIT ? 0.125f : 0.25f;
    f[0] = pack8(h);
    f[1] = pack8(h + 8);
    f[2] = pack8(s);
    f[3] = pack8(s + 8);
    if constexpr (TRAIN) {
        if (r < N) {
            bf16_t* x = X + (size_t)r * 128 + 8 * q;
            st8(x, f[0]);
            st8(x + 32, f[1]);
            st8(x + 64, f[2]);
            st8(x + 96, f[3]);
        }
    }
#pragma unroll
    for (int k = 0; k < 4; k++) f[k] = to_product(f[k], lane);
    if constexpr (LIT) {
        f[4] = flip8(f[0]);
        f[5] = flip8(f[1]);
    }
    __syncthreads();   // (the staged weights)
    product<KS>(h, sW, 0, f, lane);
    from_product(h, lane);
    ld_row<true>(b, bias, q);
    uint32_t lo = 0, hi = 0;   // one bit per column
#pragma unroll
    for (int i = 0; i < 16; i++) {
        h[i] = fmaxf(h[i] + b[i], 0.f);
        (i < 8 ? lo : hi) |= h[i] > 0.f ? 1u << (16 * (i >> 2 & 1) + (i & 3)) : 0u;
    }
    if constexpr (TRAIN) {
        lo = quad_or(lo << 4 * q);
        hi = quad_or(hi << 4 * q);
        if (r < N && q == 0) mask[r] = uint2{lo, hi};
    }
    if (r < N) st_row(H + (size_t)r * HID, h, q);
}

// One half round backward, whole, 16 rows per wavefront: with dH' = S + scale * sum of the
// neighbours' message gradients G (either may be absent: SELF, GATHER), dP = dH' * [H' > 0]
// (kept in BF16 for the weight gradient; its FP32 sum is the bias gradient) and dX = dP W: the
// columns of this row's own H go to S in place (LIT: plus those the other polarity's row has for
// it, exchanged between neighbouring lanes), the message columns to M.
// NT (see layer_bwd): S is read once a round, a round after it was written, and passes the caches.
// In the first round (LAST) what remains is the gradient of the embeddings, and dX is summed
// here instead of stored: H_l^0 = occ(l)/8 u_l + v_l, so the own columns of a literal enter the
// gradients of (u_l, v_l) with weights (occ(l)/8, 1), those of a clause (u_c, v_c) with
// (len/4, 1), and a clause's message columns, a quarter of which goes to each of its literals,
// (u_l, v_l) with (sum of occ(l)/8, len) / 4 -- a kernel that gathered them to the literals
// again took 88 us, and the rows' stores 50, of 1.94 ms.
// part: the workgroup's bias sums, 64 floats; part_e: those for u_l, v_l, u_c, v_c, 256.
template <bool LIT, bool SELF, bool GATHER, bool LAST, bool NT>
__global__ __launch_bounds__(64 * (LAST ? LAST_WAVES : LAYER_WAVES), 4) void k_layer_bwd(const int32_t* __restrict__ off, const int32_t* __restrict__ edges,
                                                      const int32_t* __restrict__ n_off, int N,
                                                      const bf16_t* __restrict__ Wt, const uint2* __restrict__ mask, const float* __restrict__ G,
                                                      float* S, bf16_t* __restrict__ dP, float* __restrict__ M,
                                                      float* __restrict__ part, float* __restrict__ part_e)
{
    constexpr int K = LIT ? 192 : 128, NW = LAST ? LAST_WAVES : LAYER_WAVES;
    __shared__ __align__(16) bf16_t sW[K * (64 + 8)];
    __shared__ float red[64 * NW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q = lane & 3;
    const int block = xcd_block(), r = 16 * (block * NW + wave) + (lane >> 2), row = min(r, N - 1);
    float* pe = part_e + (size_t)block * O_WC;
    Edges E;
    if constexpr (GATHER || LAST) E.offsets(off, row, q);
    stage_weights<K, 64>(sW, Wt);
    const int deg = GATHER || LAST ? E.e1 - E.e0 : 0;
    if constexpr (GATHER) E.ids(edges, E.e0, q);
    const uint2 m2 = r < N ? mask[row] : uint2{0u, 0u};
    const uint32_t m = (m2.x >> 8 * q & 0xFF) | (m2.y >> 8 * q & 0xFF) << 8;
    float g[16], s[16];
    if constexpr (SELF)
        ld_row<false, GATHER && NT>(g, S + (size_t)row * HID, q);   // (without GATHER S was just written)
    else {
#pragma unroll
        for (int i = 0; i < 16; i++) g[i] = 0.f;
    }
    if constexpr (GATHER) {
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = 0.f;
        gather_row(s, edges, E, q, G);
#pragma unroll
        for (int i = 0; i < 16; i++) g[i] += (LIT ? 0.25f : 0.125f) * s[i];
    }
#pragma unroll
    for (int i = 0; i < 16; i++) g[i] = m >> i & 1 ? g[i] : 0.f;
    block_sum<false>(g, red, part + (size_t)block * 64, lane, wave);   // (its barriers: the staged weights too)
    bf16x8 f[2] = {pack8(g), pack8(g + 8)};
    if (r < N) {
        st8(dP + (size_t)r * HID + 8 * q, f[0]);
        st8(dP + (size_t)r * HID + 32 + 8 * q, f[1]);
    }
    f[0] = to_product(f[0], lane);
    f[1] = to_product(f[1], lane);
    product<2>(g, sW, 1, f, lane);
    from_product(g, lane);
    if constexpr (LAST && !LIT) {
        // (a row past N has dP = 0, so dX = 0)
        int occ = 0;
        for (int e = E.e0 + q; e < E.e1; e += 4) {
            const int l = edges[e];
            occ += n_off[l + 1] - n_off[l];
        }
        occ += __builtin_amdgcn_mov_dpp(occ, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
        occ += __builtin_amdgcn_mov_dpp(occ, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
#pragma unroll
        for (int i = 0; i < 16; i++) s[i] = (float)occ * 0.03125f * g[i];
        block_sum<true>(s, red, pe, lane, wave);
#pragma unroll
        for (int i = 0; i < 16; i++) g[i] *= (float)deg * 0.25f;
        block_sum<true>(g, red, pe + O_VL, lane, wave);
    }
    if (r < N && (LIT || !LAST)) st_row(M + (size_t)r * HID, g, q);
    product<2>(g, sW, 0, f, lane);
    if constexpr (LIT) {
        product<2>(s, sW, 2, f, lane);
#pragma unroll
        for (int i = 0; i < 16; i++) g[i] += flip1(s[i]);
    }
    from_product(g, lane);
    if constexpr (LAST) {
        block_sum<true>(g, red, pe + (LIT ? O_VL : O_VC), lane, wave);
#pragma unroll
        for (int i = 0; i < 16; i++) g[i] *= (float)deg * (LIT ? 0.125f : 0.25f);
        block_sum<true>(g, red, pe + (LIT ? O_UL : O_UC), lane, wave);
        if (LIT && threadIdx.x < 128) pe[O_UC + threadIdx.x] = 0.f;
    } else if (r < N)
        st_row<NT>(S + (size_t)r * HID, g, q);
}

// Readout of 16 variables per wavefront and tile: R = relu([H_{2v+1} | H_{2v}] W_o^T + b_o),
// Y = R W_y^T + b_y (W_y in BF16); TRAIN: also the loss, dY, dP_o = (dY W_y) * [R > 0] and the
// gradient of H (S), with Z and dP_o kept in BF16 for the gradient of W_o and this
// workgroup's sums for b_o, W_y, b_y (laid out as the parameters are) and the loss.
constexpr int HEAD_PART = 256, HEAD_GRADS = O_BY + 2 - O_BO;
template <bool TRAIN>
__global__ __launch_bounds__(256) void k_readout(int V, int tiles_per_wave, const float* __restrict__ H,
                                                 const bf16_t* __restrict__ Wo, const bf16_t* __restrict__ Wot,
                                                 const bf16_t* __restrict__ Wyq, const float* __restrict__ th,
                                                 float* __restrict__ Y, const float* __restrict__ target,
                                                 const float* __restrict__ phase, const float* __restrict__ mask,
                                                 float alpha, bf16_t* __restrict__ Z, bf16_t* __restrict__ dP,
                                                 float* __restrict__ S, float* __restrict__ part)
{
    __shared__ __align__(16) bf16_t sW[64 * (128 + 8)];
    __shared__ __align__(16) bf16_t sWt[TRAIN ? 128 * (64 + 8) : 8];
    constexpr int SP = 64 + 8;
    __shared__ __align__(16) bf16_t sP[TRAIN ? 64 * SP : 8];
    __shared__ float red[256];
    stage_weights<64, 128>(sW, Wo);
    if constexpr (TRAIN) stage_weights<128, 64>(sWt, Wot);
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q = lane & 3;
    const int block = xcd_block(), t0 = (block * 4 + wave) * tiles_per_wave;
    float w0[16], w1[16], gb[16], gw0[16], gw1[16], lsum = 0.f, gy0 = 0.f, gy1 = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int d = 16 * (i >> 2) + 4 * q + (i & 3);
        w0[i] = from_bf16(Wyq[d]);
        w1[i] = from_bf16(Wyq[64 + d]);
        gb[i] = gw0[i] = gw1[i] = 0.f;
    }
    for (int t = t0; t < t0 + tiles_per_wave && 16 * t < V; t++) {
        const int v = 16 * t + (lane >> 2), row = min(v, V - 1);
        float x[16], b[16];
        bf16x8 f[4];
        ld_row(x, H + (size_t)(2 * row + 1) * HID, q);
        f[0] = pack8(x);
        f[1] = pack8(x + 8);
        ld_row(x, H + (size_t)(2 * row) * HID, q);
        f[2] = pack8(x);
        f[3] = pack8(x + 8);
        if constexpr (TRAIN) {
            if (v < V) {
                bf16_t* z = Z + (size_t)v * 128 + 8 * q;
                st8(z, f[0]);
                st8(z + 32, f[1]);
                st8(z + 64, f[2]);
                st8(z + 96, f[3]);
            }
        }
#pragma unroll
        for (int k = 0; k < 4; k++) f[k] = to_product(f[k], lane);
        product<4>(x, sW, 0, f, lane);
        from_product(x, lane);
        ld_row<true>(b, th + O_BO, q);
        float y0 = 0.f, y1 = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            x[i] = fmaxf(x[i] + b[i], 0.f);
            y0 += x[i] * w0[i];
            y1 += x[i] * w1[i];
        }
        y0 += __shfl_xor(y0, 1);
        y1 += __shfl_xor(y1, 1);
        y0 += __shfl_xor(y0, 2);
        y1 += __shfl_xor(y1, 2);
        y0 += th[O_BY];
        y1 += th[O_BY + 1];
        if (q == 0 && v < V) *reinterpret_cast<float2*>(Y + 2 * (size_t)v) = make_float2(y0, y1);
        if constexpr (TRAIN) {
            const float tg = target[row], p = phase[row], mk = mask[row];
            const float sig = 1.0f / (1.0f + expf(-y1));
            const float bce = fmaxf(y1, 0.f) - y1 * p + log1pf(expf(-fabsf(y1)));
            const bool live = v < V;
            const float da = live ? 2.0f * (y0 - tg) / (float)V : 0.f;
            const float db = live ? alpha * mk * (sig - p) / (float)V : 0.f;
            if (q == 0 && live) {
                lsum += ((y0 - tg) * (y0 - tg) + alpha * mk * bce) / (float)V;
                gy0 += da;
                gy1 += db;
            }
#pragma unroll
            for (int i = 0; i < 16; i++) {
                if (live) {
                    gw0[i] += da * x[i];
                    gw1[i] += db * x[i];
                }
                x[i] = live && x[i] > 0.f ? da * w0[i] + db * w1[i] : 0.f;
                gb[i] += x[i];
            }
            // dP is in columns out(i); the product and the stored row take in(i): through LDS
            const bf16x8 o[2] = {pack8(x), pack8(x + 8)};
            const uint4 w[2] = {__builtin_bit_cast(uint4, o[0]), __builtin_bit_cast(uint4, o[1])};
            bf16_t* tile = sP + wave * 16 * SP;
#pragma unroll
            for (int k = 0; k < 4; k++)
                *reinterpret_cast<uint2*>(tile + (lane >> 2) * SP + 16 * k + 4 * q) =
                    k & 1 ? uint2{w[k >> 1].z, w[k >> 1].w} : uint2{w[k >> 1].x, w[k >> 1].y};
            wave_sync();
            if (live) {
                st8(dP + (size_t)v * HID + 8 * q, ld8(tile + (lane >> 2) * SP + 8 * q));
                st8(dP + (size_t)v * HID + 32 + 8 * q, ld8(tile + (lane >> 2) * SP + 32 + 8 * q));
            }
            const bf16x8 g[2] = {ld8(tile + (lane & 15) * SP + 8 * (lane >> 4)),
                                 ld8(tile + (lane & 15) * SP + 32 + 8 * (lane >> 4))};
            wave_sync();
            product<2>(x, sWt, 0, g, lane);
            from_product(x, lane);
            if (live) st_row(S + (size_t)(2 * v + 1) * HID, x, q);
            product<2>(x, sWt, 1, g, lane);
            from_product(x, lane);
            if (live) st_row(S + (size_t)(2 * v) * HID, x, q);
        }
    }
    if constexpr (TRAIN) {
        float* o = part + (size_t)block * HEAD_PART;
        block_sum<true>(gb, red, o, lane, wave);
        block_sum<true>(gw0, red, o + (O_WY - O_BO), lane, wave);
        block_sum<true>(gw1, red, o + (O_WY - O_BO) + 64, lane, wave);
        gy0 = row_sum(gy0);
        gy1 = row_sum(gy1);
        lsum = row_sum(lsum);
        __syncthreads();
        if (lane == 0) {
            red[wave] = gy0;
            red[4 + wave] = gy1;
            red[8 + wave] = lsum;
        }
        __syncthreads();
        if (threadIdx.x < 64) {
            const int k = threadIdx.x;
            o[(O_BY - O_BO) + k] = k < 3 ? (red[4 * k] + red[4 * k + 1]) + (red[4 * k + 2] + red[4 * k + 3]) : 0.f;
        }
    }
}

// gfx950's transposing LDS read: within each 16-lane group, lane i receives element i % 4 of
// the 8-byte chunks that lanes i/4, i/4 + 4, i/4 + 8 and i/4 + 12 address.  With lane L of
// the group pointing at row L/4, columns 4(L%4) .. 4(L%4)+3 of a row-major 4 x 16 tile, lane
// i receives column i of those 4 rows.  Two reads (rows r .. r+3, r+4 .. r+7) give the 8
// consecutive-k values of an MFMA operand from a tile stored with k as its row index.
typedef short v4s __attribute__((ext_vector_type(4)));
__device__ __forceinline__ bf16x8 ld8_tr(const bf16_t* p, int row_stride)
{
    typedef __attribute__((address_space(3))) v4s lds_v4s;
    const v4s r0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)p);
    const v4s r1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(p + 4 * row_stride));
    typedef short v8s __attribute__((ext_vector_type(8)));
    const v8s v = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
    return __builtin_bit_cast(bf16x8, v);
}

// Partial weight gradient of this workgroup: part[blockIdx.x][64 x K] = sum over its 64-row
// chunks of dP[N x 64]^T X[N x K], N the rows of all rounds (the reduction adds the
// workgroups' partials in order).  X holds 128 columns a row; for K = 192 the other 64 are the
// first 64 of row n ^ 1.  A chunk is staged row-major in LDS (rows padded by 32 bytes) by all
// four wavefronts while the next chunk's reads are in flight, and the MFMA operands, whose k
// index is the row, come out of it through transposing reads; wavefront w computes output rows
// h = 16w .. 16w+15.
template <int K>
__global__ __launch_bounds__(256) void k_dense_dw(const bf16_t* __restrict__ dP, const bf16_t* __restrict__ X,
                                                  float* __restrict__ part, int64_t N)
{
    constexpr int SP = 64 + 16, SX = 128 + 16, CT = K / 16;   // row strides (elements) of the staged tiles
    __shared__ __align__(16) bf16_t sP[64 * SP];
    __shared__ __align__(16) bf16_t sX[64 * SX];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    // this lane's place in a transposing read: row 8(lane/16) + (lane%16)/4 of the k block,
    // columns 4(lane%4) .. +3 of the 16-column tile
    const int tr_row = 8 * (lane >> 4) + ((lane & 15) >> 2), tr_col = 4 * (lane & 3);
    uint4 p[2], x[4];
    auto load = [&](int64_t n0) {
        const int64_t rows = N - n0;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int r = (t >> 3) + 32 * k;
            p[k] = uint4{0u, 0u, 0u, 0u};
            if (r < rows) p[k] = *reinterpret_cast<const uint4*>(dP + (size_t)(n0 + r) * 64 + 8 * (t & 7));
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int r = (t >> 4) + 16 * k;
            x[k] = uint4{0u, 0u, 0u, 0u};
            if (r < rows) x[k] = *reinterpret_cast<const uint4*>(X + (size_t)(n0 + r) * 128 + 8 * (t & 15));
        }
    };
    f32x4 acc[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ct++) acc[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
    int64_t n0 = (int64_t)blockIdx.x * 64;
    const int64_t step = (int64_t)gridDim.x * 64;
    if (n0 < N) load(n0);
    for (; n0 < N; n0 += step) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 2; k++) *reinterpret_cast<uint4*>(sP + ((t >> 3) + 32 * k) * SP + 8 * (t & 7)) = p[k];
#pragma unroll
        for (int k = 0; k < 4; k++) *reinterpret_cast<uint4*>(sX + ((t >> 4) + 16 * k) * SX + 8 * (t & 15)) = x[k];
        __syncthreads();
        if (n0 + step < N) load(n0 + step);
#pragma unroll
        for (int s = 0; s < 64; s += 32) {
            // A[h][n] = dP[n][h] (16 h x 32 n), B[n][col] = X[n][col] (32 n x 16 col)
            const bf16x8 a = ld8_tr(sP + (s + tr_row) * SP + 16 * wave + tr_col, SP);
#pragma unroll
            for (int ct = 0; ct < CT; ct++) {
                const int r = ct < 8 ? s + tr_row : s + (tr_row ^ 1), c = ct < 8 ? 16 * ct : 16 * (ct - 8);
                acc[ct] = mfma32(a, ld8_tr(sX + r * SX + c + tr_col, SX), acc[ct]);
            }
        }
    }
    float* out = part + (size_t)blockIdx.x * 64 * K;
    const int dq = 4 * (lane >> 4);
#pragma unroll
    for (int ct = 0; ct < CT; ct++) {
        const int col = ct * 16 + (lane & 15);
#pragma unroll
        for (int j = 0; j < 4; j++) out[(wave * 16 + dq + j) * K + col] = acc[ct][j];
    }
}

__device__ __forceinline__ void fma4(float4& s, float a, const float4& x)
{
    s.x += a * x.x;
    s.y += a * x.y;
    s.z += a * x.z;
    s.w += a * x.w;
}
// Fixed-order reductions of the workgroups' partials, all of a pass's in two launches: every
// gradient and the loss are summed this way, never with floating-point atomics, so a gradient
// is the same bit for bit on every run.  Job: `slots` rows of `quads` float4; stage 1 splits
// the slots into `groups` contiguous runs (16 column quads x 16 interleaved slots per
// workgroup), stage 2 adds the groups in order and writes the first n floats to out and the
// rest, if out2 is given, to out2.
struct RedJob {
    const float* part;
    float* part2;
    float* out;
    float* out2;
    int slots, quads, groups, n;
};
constexpr int RED_JOBS = 8;
struct RedJobs {
    RedJob j[RED_JOBS];
    int count;
};
__global__ __launch_bounds__(256) void k_reduce_groups(RedJobs jobs)
{
    __shared__ float4 sh[16][16];
    int b = blockIdx.x, k = 0;
    for (; k < jobs.count - 1; k++) {
        const int nb = jobs.j[k].quads / 16 * jobs.j[k].groups;
        if (b < nb) break;
        b -= nb;
    }
    const RedJob& J = jobs.j[k];
    const int nx = J.quads / 16, group = b / nx, quad = 16 * (b % nx) + (threadIdx.x & 15), sub = threadIdx.x >> 4;
    if (group >= J.groups) return;
    const int per = (J.slots + J.groups - 1) / J.groups, k1 = min(J.slots, (group + 1) * per);
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
    for (int i = group * per + sub; i < k1; i += 16) fma4(s, 1.f, reinterpret_cast<const float4*>(J.part)[(size_t)i * J.quads + quad]);
    sh[sub][threadIdx.x & 15] = s;
    __syncthreads();
    if (sub == 0) {
        for (int i = 1; i < 16; i++) fma4(s, 1.f, sh[i][threadIdx.x]);
        reinterpret_cast<float4*>(J.part2)[(size_t)group * J.quads + quad] = s;
    }
}
__global__ __launch_bounds__(256) void k_reduce_final(RedJobs jobs)
{
    int b = blockIdx.x, k = 0;
    for (; k < jobs.count - 1; k++) {
        const int nb = (4 * jobs.j[k].quads + 255) / 256;
        if (b < nb) break;
        b -= nb;
    }
    const RedJob& J = jobs.j[k];
    const int i = 256 * b + threadIdx.x;
    if (i >= 4 * J.quads) return;
    float s = 0.f;
#pragma unroll 4
    for (int g = 0; g < J.groups; g++) s += J.part2[(size_t)g * 4 * J.quads + i];
    if (i < J.n)
        J.out[i] = s;
    else if (J.out2)
        J.out2[i - J.n] = s;
}

// BF16 copies of the weights: as they are (forward) and transposed (backward)
__global__ void k_quantize(const float* __restrict__ th, bf16_t* __restrict__ Wc, bf16_t* __restrict__ Wl,
                           bf16_t* __restrict__ Wo, bf16_t* __restrict__ Wct, bf16_t* __restrict__ Wlt,
                           bf16_t* __restrict__ Wot, bf16_t* __restrict__ Wy)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < 64 * 192; i += gridDim.x * blockDim.x) {
        Wl[i] = Wlt[(i % 192) * 64 + i / 192] = to_bf16(th[O_WL + i]);
        if (i < 64 * 128) {
            Wc[i] = Wct[(i % 128) * 64 + i / 128] = to_bf16(th[O_WC + i]);
            Wo[i] = Wot[(i % 128) * 64 + i / 128] = to_bf16(th[O_WO + i]);
        }
        if (i < 128) Wy[i] = to_bf16(th[O_WY + i]);
    }
}

// The incidence structure of a batch, both ways, one workgroup of 4 wavefronts per instance:
// c_off / c_edges (a clause's literal nodes, in clause order) are the arena's offsets and
// literals renumbered, l_off / l_edges (a literal's clauses, ascending) a stable counting sort
// of the edges by literal.  Each wavefront takes a contiguous quarter of the instance's edges
// with its own counters (cnt[w][l], LDS); the places of equal literals within 64 edges follow
// from matching their codes bit by bit with ballots, so the order is that of a serial pass.
// Built on the host this took 1.3 ms, and its copies 0.35 ms, of the 2.4 ms of an inference on
// 256 x (n=300, m=1278).
// clause_of: scratch, one int per edge.  Limits (see gnn_graph_on_device): the counters fit 64 KB
// of LDS, and no clause is so long that one thread listing it is what takes the time.
constexpr int GRAPH_WAVES = 4;
__global__ __launch_bounds__(64 * GRAPH_WAVES) void k_graph(const InstMeta* __restrict__ meta, const int32_t* __restrict__ lits,
                                                            const int32_t* __restrict__ coff,
                                                            const int32_t* __restrict__ var_base, int n_inst,
                                                            int32_t* __restrict__ clause_of, int32_t* __restrict__ c_off,
                                                            int32_t* __restrict__ c_edges, int32_t* __restrict__ l_off,
                                                            int32_t* __restrict__ l_edges)
{
    extern __shared__ int cnt[];
    __shared__ int sums[64 * GRAPH_WAVES];
    const int inst = blockIdx.x, t = threadIdx.x, nt = 64 * GRAPH_WAVES;
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const InstMeta mi = meta[inst];
    const int m = mi.m, L = 2 * mi.n, l0 = 2 * var_base[inst], c0 = (int)(mi.coff_base - inst), e0 = (int)mi.lit_base;
    const int32_t* co = coff + mi.coff_base;
    const int E = co[m];
    for (int i = t; i < GRAPH_WAVES * L; i += nt) cnt[i] = 0;
    if (inst == 0 && t == 0) c_off[0] = 0;
    for (int c = t; c < m; c += nt) {
        const int k1 = co[c + 1];
        c_off[c0 + c + 1] = e0 + k1;
        for (int k = co[c]; k < k1; k++) clause_of[e0 + k] = c0 + c;
    }
    for (int k = t; k < E; k += nt) c_edges[e0 + k] = l0 + lits[e0 + k];
    __syncthreads();
    // counts
    int* my = cnt + wave * L;
    const int per = (E + nt - 1) / nt * 64;
    const int k0 = min(E, wave * per), k1 = min(E, k0 + per);
    for (int k = k0 + lane; k < k1; k += 64) atomicAdd(&my[lits[e0 + k]], 1);
    __syncthreads();
    // exclusive prefix over (literal, wavefront): each thread takes a run of literals
    const int run = (L + nt - 1) / nt, a = min(L, t * run), b = min(L, a + run);
    int sum = 0;
    for (int l = a; l < b; l++)
        for (int w = 0; w < GRAPH_WAVES; w++) sum += cnt[w * L + l];
    sums[t] = sum;
    __syncthreads();
    for (int o = 1; o < nt; o <<= 1) {
        const int v = t >= o ? sums[t - o] : 0;
        __syncthreads();
        sums[t] += v;
        __syncthreads();
    }
    int at = e0 + sums[t] - sum;
    for (int l = a; l < b; l++) {
        l_off[l0 + l] = at;
        for (int w = 0; w < GRAPH_WAVES; w++) {
            const int c = cnt[w * L + l];
            cnt[w * L + l] = at;
            at += c;
        }
    }
    if (inst == n_inst - 1 && t == 0) l_off[l0 + L] = e0 + E;
    __syncthreads();
    // placement
    const int bits = L > 1 ? 32 - __clz(L - 1) : 0;
    for (int kb = k0; kb < k1; kb += 64) {
        const int k = kb + lane;
        const bool live = k < k1;
        const int l = live ? lits[e0 + k] : 0, c = live ? clause_of[e0 + k] : 0;
        uint64_t same = ballot(live);
        for (int i = 0; i < bits; i++) {
            const uint64_t v = ballot(l >> i & 1);
            same &= l >> i & 1 ? v : ~v;
        }
        const int pos = my[l] + __popcll(same & ((1ull << lane) - 1ull));
        wave_sync();
        if (live) {
            l_edges[pos] = c;
            if (same >> lane == 1ull) my[l] = pos + 1;   // the last of its literal
        }
        wave_sync();
    }
}

__global__ void k_adam(float* __restrict__ th, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v,
                       int n, float lr, float b1, float b2, float eps, float c1, float c2)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.f - b1) * gi;
        const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        th[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    }
}

}  // namespace gnn
}  // namespace gpsat

// ---------------------------------------------------------------------------------------
// Host orchestration and C ABI.
using namespace gpsat;
using namespace gpsat::gnn;

// Workgroups of the weight-gradient products (one partial matrix each; two workgroups per CU, as
// more of them write more partials and gain nothing).
constexpr int DW_BLOCKS = 512;
constexpr int MAX_GROUPS = 32;

// One pass's activations, carved from the model's arena (see gpsat_gnn_model); the second part
// only for a pass with gradients.
struct Acts {
    float *Hl = nullptr, *Hc = nullptr;
    bf16_t *Xc = nullptr, *Xl = nullptr, *Z = nullptr;                        // [rounds][rows][128]
    bf16_t *dPc = nullptr, *dPl = nullptr, *dPo = nullptr;                    // [rounds][rows][64]
    uint2 *mask_c = nullptr, *mask_l = nullptr;                               // [rounds][rows]
    float *Sl = nullptr, *Ml = nullptr, *Sc = nullptr, *Mc = nullptr, *loss = nullptr;
    float *part_o = nullptr, *part_l = nullptr, *part_c = nullptr, *part_e = nullptr;
    float *part_wl = nullptr, *part_wc = nullptr, *part_wo = nullptr, *part2 = nullptr;
};

// A model: FP32 master parameters, gradient, Adam moments, BF16 weight copies, and a grow-only
// arena that holds the activations and gradient partials of the pass being run.  Graphs own
// only their incidence structure and labels, so a training loop keeps every batch's graph
// across steps without holding every batch's activations; calls on one model therefore run
// one at a time.
struct gpsat_gnn_model {
    float* th = nullptr;
    float* grad = nullptr;
    float* m = nullptr;
    float* v = nullptr;
    bf16_t *Wc = nullptr, *Wl = nullptr, *Wo = nullptr, *Wy = nullptr;
    bf16_t *Wct = nullptr, *Wlt = nullptr, *Wot = nullptr;
    char* arena = nullptr;
    size_t arena_bytes = 0;
    int64_t step = 0;
    bool dirty = true;
};

// A graph's arrays are pieces of one block of the device-memory cache (devmem_cache_*), which
// takes it back once the graph's stream is idle.  The stream is created and destroyed with the
// graph (~75 us): kept for the next graph it would hold a hardware queue meanwhile, and two
// batches evaluated at the same time then shared one (31 -> 43 us a pass).
struct gpsat_gnn_graph {
    int32_t V = 0, L = 0, C = 0, R = 3;
    int64_t E = 0;
    int32_t *c_off = nullptr, *c_edges = nullptr, *l_off = nullptr, *l_edges = nullptr;
    float *Y = nullptr, *target = nullptr, *phase = nullptr, *mask = nullptr;
    int32_t *clause_of = nullptr, *var_base = nullptr;   // k_graph's
    hipStream_t st = nullptr;
    int dev = 0;
    void* block = nullptr;
    size_t block_bytes = 0;
    ~gpsat_gnn_graph()
    {
        const bool idle = st && hipStreamSynchronize(st) == hipSuccess;
        if (block && !(idle && devmem_cache_give(dev, block, block_bytes))) (void)hipFree(block);
        if (st) (void)hipStreamDestroy(st);
    }
    // the pieces, laid out in `base` (nullptr: only count); returns the bytes used
    size_t carve(char* base, int32_t n_inst)
    {
        size_t off = 0;
        auto take = [&](auto*& p, size_t count) {
            using T = std::remove_reference_t<decltype(*p)>;
            p = base ? (T*)(base + off) : nullptr;
            off += (std::max<size_t>(count, 1) * sizeof(T) + 255) & ~(size_t)255;
        };
        take(c_off, (size_t)C + 1);
        take(c_edges, E);
        take(l_off, (size_t)L + 1);
        take(l_edges, E);
        take(Y, (size_t)V * 2);
        take(target, V);
        take(phase, V);
        take(mask, V);
        take(clause_of, E);
        take(var_base, n_inst);
        return off;
    }
    hipError_t alloc(int32_t n_inst)
    {
        hipError_t e = hipGetDevice(&dev);
        if (e == hipSuccess) e = hipStreamCreateWithFlags(&st, hipStreamNonBlocking);
        if (e != hipSuccess) return e;
        const size_t bytes = devmem_round(carve(nullptr, n_inst));
        block = devmem_cache_take(dev, bytes);
        if (!block) e = hipMalloc(&block, bytes);
        if (e != hipSuccess) {
            block = nullptr;
            return e;
        }
        block_bytes = bytes;
        carve((char*)block, n_inst);
        return hipSuccess;
    }
};

#define GNN_TRY(expr)                                                              \
    do {                                                                           \
        hipError_t _e = (expr);                                                    \
        if (_e != hipSuccess) {                                                    \
            set_error(std::string(#expr) + ": " + hipGetErrorString(_e));          \
            return _e == hipErrorOutOfMemory ? GPSAT_ERR_NOMEM : GPSAT_ERR_HIP;    \
        }                                                                          \
    } while (0)

namespace {

// Workgroups that cover N rows, 16 * tiles each: a multiple of 8, see xcd_block.
int row_blocks(int64_t N, int tiles) { return (int)(((N + 16 * tiles - 1) / (16 * tiles) + 7) / 8 * 8); }
// Bias partials of a layer over N rows: the first round's workgroups, then the other rounds'.
size_t bias_slot(int64_t N, int t) { return t ? row_blocks(N, LAST_WAVES) + (size_t)(t - 1) * row_blocks(N, LAYER_WAVES) : 0; }
// The readout's wavefronts take several tiles in turn where there are enough to fill the GPU:
// both forms of W_o are staged per workgroup.
int readout_tiles(int V) { return std::max(1, std::min(4, V / (16 * 2048))); }
int dw_blocks(int64_t rows) { return (int)std::max<int64_t>(1, std::min<int64_t>(DW_BLOCKS, (rows + 63) / 64)); }
int red_groups(int64_t slots) { return (int)std::max<int64_t>(1, std::min<int64_t>(MAX_GROUPS, slots / 64)); }

// Lay a pass's activations out in `base` (nullptr: only count); returns the bytes used.
// Every piece starts 256-byte aligned.
size_t carve(const gpsat_gnn_graph* g, bool train, char* base, Acts& a)
{
    size_t off = 0;
    auto take = [&](auto*& p, size_t count) {
        using T = std::remove_reference_t<decltype(*p)>;
        p = base ? (T*)(base + off) : nullptr;
        off += (std::max<size_t>(count, 1) * sizeof(T) + 255) & ~(size_t)255;
    };
    const size_t L = g->L, C = g->C, V = g->V, R = g->R;
    take(a.Hl, L * HID);
    take(a.Hc, C * HID);
    if (!train) return off;
    take(a.Xc, R * C * 128);
    take(a.Xl, R * L * 128);
    take(a.Z, V * 128);
    take(a.dPc, R * C * HID);
    take(a.dPl, R * L * HID);
    take(a.dPo, V * HID);
    take(a.mask_c, R * C);
    take(a.mask_l, R * L);
    take(a.Sl, L * HID);
    take(a.Ml, L * HID);
    take(a.Sc, C * HID);
    take(a.Mc, C * HID);
    take(a.loss, HEAD_PART - HEAD_GRADS);   // (the rest of a readout partial's row)
    take(a.part_o, (size_t)row_blocks(V, 4 * readout_tiles((int)V)) * HEAD_PART);
    take(a.part_l, bias_slot(L, (int)R) * HID);
    take(a.part_c, bias_slot(C, (int)R) * HID);
    take(a.part_e, ((size_t)row_blocks(L, LAST_WAVES) + row_blocks(C, LAST_WAVES)) * O_WC);   // literals' workgroups, then clauses'
    take(a.part_wl, (size_t)dw_blocks(R * L) * 64 * 192);
    take(a.part_wc, (size_t)dw_blocks(R * C) * 64 * 128);
    take(a.part_wo, (size_t)dw_blocks(V) * 64 * 128);
    take(a.part2, (size_t)MAX_GROUPS * (HEAD_PART + 6 * HID + 64 * (192 + 128 + 128)));
    return off;
}

// The activations of a pass of graph g in model m's arena (grown if it needs more).
hipError_t acts_for(gpsat_gnn_model* m, gpsat_gnn_graph* g, bool train, Acts& a)
{
    const size_t need = carve(g, train, nullptr, a);
    if (need > m->arena_bytes) {
        hipError_t e = hipDeviceSynchronize();
        if (e != hipSuccess) return e;
        (void)hipFree(m->arena);
        m->arena = nullptr;
        m->arena_bytes = 0;
        e = hipMalloc(&m->arena, need);
        if (e != hipSuccess) return e;
        m->arena_bytes = need;
    }
    carve(g, train, m->arena, a);
    return hipSuccess;
}

template <bool LIT, bool FIRST, bool TRAIN>
void layer(gpsat_gnn_model* m, gpsat_gnn_graph* g, const Acts& a, int t)
{
    const int N = LIT ? g->L : g->C;
    if (N == 0) return;
    hipLaunchKernelGGL((k_layer<LIT, FIRST, TRAIN>), dim3(row_blocks(N, LAYER_WAVES)), dim3(64 * LAYER_WAVES), 0, g->st,
                       LIT ? g->l_off : g->c_off, LIT ? g->l_edges : g->c_edges, LIT ? g->c_off : g->l_off, N, m->th,
                       LIT ? m->Wl : m->Wc, m->th + (LIT ? O_BL : O_BC), LIT ? a.Hc : a.Hl, LIT ? a.Hl : a.Hc,
                       TRAIN ? (LIT ? a.Xl : a.Xc) + (size_t)t * N * 128 : nullptr,
                       TRAIN ? (LIT ? a.mask_l : a.mask_c) + (size_t)t * N : nullptr);
}

// Forward pass, readout included (TRAIN: with the loss and the readout's gradients).
template <bool TRAIN>
hipError_t forward_pass(gpsat_gnn_model* m, gpsat_gnn_graph* g, const Acts& a, float alpha)
{
    if (m->dirty) {
        hipLaunchKernelGGL(k_quantize, dim3(48), dim3(256), 0, g->st, m->th, m->Wc, m->Wl, m->Wo, m->Wct, m->Wlt, m->Wot,
                           m->Wy);
        m->dirty = false;
    }
    layer<false, true, TRAIN>(m, g, a, 0);
    layer<true, true, TRAIN>(m, g, a, 0);
    for (int t = 1; t < g->R; t++) {
        layer<false, false, TRAIN>(m, g, a, t);
        layer<true, false, TRAIN>(m, g, a, t);
    }
    const int tiles = readout_tiles(g->V);
    if (g->V)
        hipLaunchKernelGGL((k_readout<TRAIN>), dim3(row_blocks(g->V, 4 * tiles)), dim3(256), 0, g->st, g->V, tiles, a.Hl, m->Wo, m->Wot,
                           m->Wy, m->th, g->Y, g->target, g->phase, g->mask, alpha, a.Z, a.dPo, a.Sl, a.part_o);
    return hipGetLastError();
}

template <bool LIT, bool SELF, bool GATHER, bool LAST>
void layer_bwd(gpsat_gnn_model* m, gpsat_gnn_graph* g, const Acts& a, int t)
{
    const int N = LIT ? g->L : g->C;
    if (N == 0) return;
    constexpr int NW = LAST ? LAST_WAVES : LAYER_WAVES;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(row_blocks(N, NW)), dim3(64 * NW), 0, g->st,
                           LIT ? g->l_off : g->c_off, LIT ? g->l_edges : g->c_edges, LIT ? g->c_off : g->l_off, N,
                           LIT ? m->Wlt : m->Wct,
                           (LIT ? a.mask_l : a.mask_c) + (size_t)t * N, LIT ? a.Mc : a.Ml, LIT ? a.Sl : a.Sc,
                           (LIT ? a.dPl : a.dPc) + (size_t)t * N * HID, LIT ? a.Ml : a.Mc,
                           (LIT ? a.part_l : a.part_c) + bias_slot(N, t) * HID,
                           a.part_e + (LIT ? 0 : (size_t)row_blocks(g->L, LAST_WAVES) * O_WC));
    };
    // Rows' gradients beyond the 256 MB last-level cache are kept out of it, which leaves it to the
    // gathered ones (961,536 rows: the pass 1.78 -> 1.75 ms); smaller ones stay (235,000 rows: 519
    // us, past the caches 529).
    if ((int64_t)(g->L + (int64_t)g->C) * 2 * HID * 4 > (int64_t)256 << 20)
        launch(k_layer_bwd<LIT, SELF, GATHER, LAST, true>);
    else
        launch(k_layer_bwd<LIT, SELF, GATHER, LAST, false>);
}

// Backward pass from the readout's gradients to m->grad (every element written) and the loss.
hipError_t backward_pass(gpsat_gnn_model* m, gpsat_gnn_graph* g, const Acts& a)
{
    hipStream_t st = g->st;
    const int R = g->R, L = g->L, C = g->C, V = g->V;
    for (int t = R - 1; t >= 0; t--) {
        const bool top = t == R - 1;
        if (top && t)
            layer_bwd<true, true, false, false>(m, g, a, t);
        else if (top)
            layer_bwd<true, true, false, true>(m, g, a, t);
        else if (t)
            layer_bwd<true, true, true, false>(m, g, a, t);
        else
            layer_bwd<true, true, true, true>(m, g, a, t);
        if (top && t)
            layer_bwd<false, false, true, false>(m, g, a, t);
        else if (top)
            layer_bwd<false, false, true, true>(m, g, a, t);
        else if (t)
            layer_bwd<false, true, true, false>(m, g, a, t);
        else
            layer_bwd<false, true, true, true>(m, g, a, t);
    }
    const int bl = dw_blocks((int64_t)R * L), bc = dw_blocks((int64_t)R * C), bo = dw_blocks(V);
    hipLaunchKernelGGL((k_dense_dw<192>), dim3(bl), dim3(256), 0, st, a.dPl, a.Xl, a.part_wl, (int64_t)R * L);
    hipLaunchKernelGGL((k_dense_dw<128>), dim3(bc), dim3(256), 0, st, a.dPc, a.Xc, a.part_wc, (int64_t)R * C);
    hipLaunchKernelGGL((k_dense_dw<128>), dim3(bo), dim3(256), 0, st, a.dPo, a.Z, a.part_wo, (int64_t)V);
    RedJobs jobs{};
    int nb1 = 0, nb2 = 0;
    float* part2 = a.part2;
    auto job = [&](const float* part, int slots, int width, float* out, int n, float* out2 = nullptr) {
        const int gr = red_groups(slots);
        jobs.j[jobs.count++] = RedJob{part, part2, out, out2, slots, width / 4, gr, n};
        part2 += (size_t)gr * width;
        nb1 += width / 64 * gr;
        nb2 += (width + 255) / 256;
    };
    job(a.part_o, V ? row_blocks(V, 4 * readout_tiles(V)) : 0, HEAD_PART, m->grad + O_BO, HEAD_GRADS, a.loss);
    job(a.part_l, (int)bias_slot(L, R), HID, m->grad + O_BL, HID);
    job(a.part_c, (int)bias_slot(C, R), HID, m->grad + O_BC, HID);
    job(a.part_e, row_blocks(L, LAST_WAVES) + row_blocks(C, LAST_WAVES), O_WC, m->grad, O_WC);
    job(a.part_wl, bl, 64 * 192, m->grad + O_WL, 64 * 192);
    job(a.part_wc, bc, 64 * 128, m->grad + O_WC, 64 * 128);
    job(a.part_wo, bo, 64 * 128, m->grad + O_WO, 64 * 128);
    hipLaunchKernelGGL(k_reduce_groups, dim3(nb1), dim3(256), 0, st, jobs);
    hipLaunchKernelGGL(k_reduce_final, dim3(nb2), dim3(256), 0, st, jobs);
    return hipGetLastError();
}

hipError_t build_on_device(gpsat_gnn_graph* g, const DeviceBatch& d, const std::vector<int32_t>& var_base)
{
    hipError_t e = hipMemcpyAsync(g->var_base, var_base.data(), 4 * (size_t)d.n_inst, hipMemcpyHostToDevice, g->st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_graph, dim3(d.n_inst), dim3(64 * GRAPH_WAVES), (size_t)GRAPH_WAVES * 2 * d.max_n * 4, g->st, d.meta,
                       d.lits, d.coff, g->var_base, d.n_inst, g->clause_of, g->c_off, g->c_edges, g->l_off, g->l_edges);
    e = hipGetLastError();
    return e == hipSuccess ? hipStreamSynchronize(g->st) : e;
}

hipError_t build_on_host(gpsat_gnn_graph* g, const DeviceBatch& d, const std::vector<int32_t>& var_base)
{
    std::vector<int32_t> c_off((size_t)g->C + 1, 0), c_edges(g->E), l_off((size_t)g->L + 1, 0), l_edges(g->E);
    int32_t cg = 0;
    for (int32_t i = 0; i < d.n_inst; i++) {
        const InstMeta& mi = d.h_meta[i];
        const int32_t* co = d.h_coff.data() + mi.coff_base;
        for (int32_t c = 0; c < mi.m; c++, cg++) {
            c_off[cg + 1] = (int32_t)(mi.lit_base + co[c + 1]);
            for (int32_t k = co[c]; k < co[c + 1]; k++) {
                const int32_t ln = 2 * var_base[i] + d.h_lits[mi.lit_base + k];
                c_edges[mi.lit_base + k] = ln;
                l_off[ln + 1]++;
            }
        }
    }
    for (int32_t l = 0; l < g->L; l++) l_off[l + 1] += l_off[l];
    std::vector<int32_t> fill(l_off.begin(), l_off.end() - 1);
    for (int32_t c = 0; c < g->C; c++)
        for (int32_t e = c_off[c]; e < c_off[c + 1]; e++) l_edges[fill[c_edges[e]]++] = c;
    hipError_t e = hipMemcpy(g->c_off, c_off.data(), 4 * c_off.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess && g->E) e = hipMemcpy(g->c_edges, c_edges.data(), 4 * g->E, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(g->l_off, l_off.data(), 4 * l_off.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess && g->E) e = hipMemcpy(g->l_edges, l_edges.data(), 4 * g->E, hipMemcpyHostToDevice);
    return e;
}

}  // namespace

extern "C" {

int gpsat_gnn_param_count(int32_t* n)
{
    if (!n) {
        set_error("null argument");
        return GPSAT_ERR_ARG;
    }
    *n = N_PARAMS;
    return GPSAT_OK;
}

int gpsat_gnn_model_create(const float* theta, gpsat_gnn_model** out)
{
    if (!out || !theta) {
        set_error("null argument");
        return GPSAT_ERR_ARG;
    }
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) {
        set_error("no HIP device visible");
        return GPSAT_ERR_NODEVICE;
    }
    gpsat_gnn_model* m = new gpsat_gnn_model();
    hipError_t e = hipMalloc(&m->th, 4 * N_PARAMS);
    if (e == hipSuccess) e = hipMalloc(&m->grad, 4 * N_PARAMS);
    if (e == hipSuccess) e = hipMalloc(&m->m, 4 * N_PARAMS);
    if (e == hipSuccess) e = hipMalloc(&m->v, 4 * N_PARAMS);
    if (e == hipSuccess) e = hipMalloc(&m->Wc, 2 * 64 * 128);
    if (e == hipSuccess) e = hipMalloc(&m->Wl, 2 * 64 * 192);
    if (e == hipSuccess) e = hipMalloc(&m->Wo, 2 * 64 * 128);
    if (e == hipSuccess) e = hipMalloc(&m->Wy, 2 * 128);
    if (e == hipSuccess) e = hipMalloc(&m->Wct, 2 * 64 * 128);
    if (e == hipSuccess) e = hipMalloc(&m->Wlt, 2 * 64 * 192);
    if (e == hipSuccess) e = hipMalloc(&m->Wot, 2 * 64 * 128);
    if (e == hipSuccess) e = hipMemcpy(m->th, theta, 4 * N_PARAMS, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(m->m, 0, 4 * N_PARAMS);
    if (e == hipSuccess) e = hipMemset(m->v, 0, 4 * N_PARAMS);
    if (e != hipSuccess) {
        set_error(std::string("gnn model: ") + hipGetErrorString(e));
        gpsat_gnn_model_destroy(m);
        return GPSAT_ERR_HIP;
    }
    *out = m;
    return GPSAT_OK;
}

int gpsat_gnn_model_destroy(gpsat_gnn_model* m)
{
    if (!m) return GPSAT_OK;
    (void)hipDeviceSynchronize();
    for (void* p : {(void*)m->th, (void*)m->grad, (void*)m->m, (void*)m->v, (void*)m->arena, (void*)m->Wc,
                    (void*)m->Wl, (void*)m->Wo, (void*)m->Wy, (void*)m->Wct, (void*)m->Wlt, (void*)m->Wot})
        (void)hipFree(p);
    delete m;
    return GPSAT_OK;
}

int gpsat_gnn_model_params(gpsat_gnn_model* m, float* theta)
{
    if (!m || !theta) {
        set_error("null argument");
        return GPSAT_ERR_ARG;
    }
    GNN_TRY(hipDeviceSynchronize());
    GNN_TRY(hipMemcpy(theta, m->th, 4 * N_PARAMS, hipMemcpyDeviceToHost));
    return GPSAT_OK;
}

int gpsat_gnn_graph_create(gpsat_batch* b, int32_t rounds, gpsat_gnn_graph** out)
{
    if (!b || !out || rounds < 1 || rounds > 16) {
        set_error("bad argument");
        return GPSAT_ERR_ARG;
    }
    *out = nullptr;
    DeviceBatch& d = b->d;
    gpsat_gnn_graph* g = new gpsat_gnn_graph();
    g->R = rounds;
    std::vector<int32_t> var_base(d.n_inst + 1, 0);
    for (int32_t i = 0; i < d.n_inst; i++) var_base[i + 1] = var_base[i] + d.h_meta[i].n;
    g->V = var_base[d.n_inst];
    g->L = 2 * g->V;
    g->C = (int32_t)d.n_clauses;
    g->E = d.n_lits;
    hipError_t e = g->alloc(d.n_inst);
    if (e == hipSuccess) e = gnn_graph_on_device(d, g->dev) ? build_on_device(g, d, var_base) : build_on_host(g, d, var_base);
    if (e != hipSuccess) {
        set_error(std::string("gnn graph: ") + hipGetErrorString(e));
        delete g;
        return e == hipErrorOutOfMemory ? GPSAT_ERR_NOMEM : GPSAT_ERR_HIP;
    }
    *out = g;
    return GPSAT_OK;
}

int gpsat_gnn_graph_destroy(gpsat_gnn_graph* g)
{
    delete g;
    return GPSAT_OK;
}

int gpsat_gnn_graph_labels(gpsat_gnn_graph* g, const float* target, const float* phase, const float* mask)
{
    if (!g || !target || !phase || !mask) {
        set_error("null argument");
        return GPSAT_ERR_ARG;
    }
    GNN_TRY(hipMemcpyAsync(g->target, target, 4 * (size_t)g->V, hipMemcpyHostToDevice, g->st));
    GNN_TRY(hipMemcpyAsync(g->phase, phase, 4 * (size_t)g->V, hipMemcpyHostToDevice, g->st));
    GNN_TRY(hipMemcpyAsync(g->mask, mask, 4 * (size_t)g->V, hipMemcpyHostToDevice, g->st));
    GNN_TRY(hipStreamSynchronize(g->st));
    return GPSAT_OK;
}

int gpsat_gnn_forward(gpsat_gnn_model* m, gpsat_gnn_graph* g, float* y)
{
    if (!m || !g || !y) {
        set_error("null argument");
        return GPSAT_ERR_ARG;
    }
    Acts a;
    GNN_TRY(acts_for(m, g, false, a));
    GNN_TRY(forward_pass<false>(m, g, a, 0.f));
    GNN_TRY(hipMemcpyAsync(y, g->Y, 8 * (size_t)g->V, hipMemcpyDeviceToHost, g->st));
    GNN_TRY(hipStreamSynchronize(g->st));
    return GPSAT_OK;
}

int gpsat_gnn_loss_grad(gpsat_gnn_model* m, gpsat_gnn_graph* g, float alpha, float* loss, float* grad, float* y)
{
    if (!m || !g) {
        set_error("null argument");
        return GPSAT_ERR_ARG;
    }
    Acts a;
    GNN_TRY(acts_for(m, g, true, a));
    GNN_TRY(forward_pass<true>(m, g, a, alpha));
    GNN_TRY(backward_pass(m, g, a));
    if (loss) GNN_TRY(hipMemcpyAsync(loss, a.loss, 4, hipMemcpyDeviceToHost, g->st));
    if (grad) GNN_TRY(hipMemcpyAsync(grad, m->grad, 4 * N_PARAMS, hipMemcpyDeviceToHost, g->st));
    if (y) GNN_TRY(hipMemcpyAsync(y, g->Y, 8 * (size_t)g->V, hipMemcpyDeviceToHost, g->st));
    GNN_TRY(hipStreamSynchronize(g->st));
    return GPSAT_OK;
}

int gpsat_gnn_train_step(gpsat_gnn_model* m, gpsat_gnn_graph* g, float alpha, float lr, float* loss)
{
    if (!m || !g || !(lr > 0.f)) {
        set_error("bad argument");
        return GPSAT_ERR_ARG;
    }
    Acts a;
    GNN_TRY(acts_for(m, g, true, a));
    GNN_TRY(forward_pass<true>(m, g, a, alpha));
    GNN_TRY(backward_pass(m, g, a));
    m->step++;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - powf(b1, (float)m->step), c2 = 1.f - powf(b2, (float)m->step);
    hipLaunchKernelGGL(k_adam, dim3(64), dim3(256), 0, g->st, m->th, m->grad, m->m, m->v, N_PARAMS, lr, b1, b2, 1e-8f,
                       c1, c2);
    m->dirty = true;
    GNN_TRY(hipGetLastError());
    if (loss) GNN_TRY(hipMemcpyAsync(loss, a.loss, 4, hipMemcpyDeviceToHost, g->st));
    GNN_TRY(hipStreamSynchronize(g->st));
    return GPSAT_OK;
}

}  // extern "C"
