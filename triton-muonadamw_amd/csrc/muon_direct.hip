// Muon step for gfx950, direct path: Newton-Schulz products whose operands go
// straight from memory to the MFMA registers, one wavefront per output tile.
//
// A product of one small matrix has few 128 x 128 tiles (21 for the Gram of a
// 768 x 3072 matrix), so the LDS-staged kernel of muon.hip leaves most CUs
// idle, and each of its workgroups moves its operands at the rate one CU gets
// from the L2 (about 27 bytes per cycle).  Here a workgroup is one wavefront
// that owns a 32 x 32 or 64 x 64 output tile and walks the whole reduction, so
// the same Gram is 300 workgroups, with no barrier and no LDS in the k loop.
// Every output element sums the same products in the same order as there (one
// v_mfma_f32_32x32x16_bf16 chain, k ascending), so the results are the same
// bits.  Measured in the step, staged -> direct: one 3072 x 768 matrix, Gram
// 28.6 -> 8.9 us, polynomial 9.9 -> 4.3, update 10.5 -> 10.6, step 269 -> 143;
// two 512 x 2048, Gram 17.8 -> 6.0, polynomial 7.6 -> 3.9, update 9.5 -> 8.6,
// step 198 -> 108.  What is left of a small launch is latency: 1.5 us for an empty kernel,
// then the arguments, the operands (written by other XCDs, so past the L2) and
// the stores, one after the other.  A larger one is bound by the L2's operand
// traffic (26 TB/s fits 460 measured steps), which the staged tiles halve: the
// host takes this path where it is the cheaper one (hip_muon.py, direct_pays).
//
// Layout of the workspace matrices (fragment-major, foff): blocks of 32 rows x
// 16 columns, 1 KB each, holding the 16 bytes lane l = 32 * (c / 8 % 2) + r % 32
// of a fragment needs at 16 * l, so that an operand load is one contiguous KB.
// (The same loads out of 128-byte rows, 16 rows to an instruction, ran at a
// quarter of the rate: lanes that follow each other must be contiguous.)
// Both X (the Gram's operand) and X^T (the update's) are kept.
//
// One launch serves up to 64 matrices of any shapes: a block finds its matrix
// in the launch's list of first blocks, and its record in a table that the
// prep kernel leaves in the workspace (4 KB of kernel argument once per step
// instead of 17 times).
//   1. direct_prep_kernel   momentum, Nesterov blend, bf16 cast into X and X^T,
//                           one sum of squares per unit of 32 x 128 elements.
//   2. direct_scale_kernel  the norm (the fixed-order sum of muon_norm_kernel,
//                           by every block) and X, X^T = bf16(. * 1/norm).
//   3. ns_steps x { Gram, polynomial, update }, the last update applying the
//      step to the parameter.
#include "mamw_device.h"
#include "mamw_launch.h"
#include "mamw_plan.h"

namespace mamw {
namespace {

enum DirectMode { DM_GRAM = 0, DM_POLY = 1, DM_UPDATE = 2, DM_APPLY = 3 };

typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4_t* lds_i16x4_ptr_t;
typedef __attribute__((address_space(3))) void* lds_ptr_t;

constexpr int kStoreThrough = 16;  // cache policy bits of a store: sc1 (agent scope, written through)

// Element offset of (r, c) in a fragment-major matrix of `rows` rows.
__device__ __forceinline__ int foff(int rows, int r, int c) {
    return (((c >> 4) * (rows >> 5) + (r >> 5)) << 9) + (((c >> 3) & 1) << 8) + ((r & 31) << 3) + (c & 7);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, int(bytes), 0x00020000);
}

// Matrix of launch block `block`: the last one whose first block is not after
// it (one entry per lane and a ballot).
__device__ __forceinline__ int find_matrix(const DirectIndex& x, int block) {
    if (x.count == 1) return 0;
    const int i = int(threadIdx.x) & 63;
    const bool le = i < x.count && x.begin[i] <= block;
    return __builtin_amdgcn_readfirstlane(int(__popcll(__ballot(le))) - 1);
}

// Entry of the launch table in the workspace: scalar loads (the table was
// written by the launch's prep kernel, before this one began).
typedef const __attribute__((address_space(4))) DirectMat* table_ptr_t;
__device__ __forceinline__ DirectMat table_entry(const char* ws, int i) {
    table_ptr_t t = (table_ptr_t)(uintptr_t)(ws);
    DirectMat d;
    d.param = t[i].param;
    d.grad = t[i].grad;
    d.mom = t[i].mom;
    d.upd = t[i].upd;
    d.rows = t[i].rows;
    d.cols = t[i].cols;
    d.mp = t[i].mp;
    d.np = t[i].np;
    d.ws = t[i].ws;
    d.slr = t[i].slr;
    d.tall = t[i].tall;
    d.flags = t[i].flags;
    return d;
}

// Blocks are dealt to the 8 XCDs round-robin; each XCD takes a contiguous
// range of the launch's tiles, whose operands its L2 then holds.
__device__ __forceinline__ int xcd_contiguous(int block, int total) {
    const int x = block & 7, q = total >> 3, r = total & 7;
    return x * q + min(x, r) + (block >> 3);
}

// A 32 x 128 tile in LDS (rows of LD halves) at (r0, c0) of an Rp x Cp matrix
// into the fragment-major `along` (same rows) and `across` (transposed), if not
// NULL: 8 blocks of 1 KB each, as far as the matrix goes.
template <int LD>
__device__ __forceinline__ void store_unit(const uint16_t* tile, int tid, int r0, int c0, int Rp, int Cp, uint16_t* along,
                                           uint16_t* across) {
    if (along) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int id = tid + 256 * k, blk = id >> 6, row = id & 31, half = (id >> 5) & 1;
            const int cc = blk * 16 + half * 8;
            if (c0 + blk * 16 < Cp)
                *reinterpret_cast<uint4*>(along + foff(Rp, r0 + row, c0 + cc)) =
                    *reinterpret_cast<const uint4*>(&tile[row * LD + cc]);
        }
    }
    if (across) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int id = tid + 256 * k, blk = id >> 6, half = (id >> 5) & 1;
            const int cl = (blk >> 1) * 32 + (id & 31), rl = (blk & 1) * 16 + half * 8;
            if (c0 + (blk >> 1) * 32 < Cp) {
                uint32_t w[4];
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    w[q] = uint32_t(tile[(rl + 2 * q) * LD + cl]) | (uint32_t(tile[(rl + 2 * q + 1) * LD + cl]) << 16);
                *reinterpret_cast<uint4*>(across + foff(Cp, c0 + cl, r0 + rl)) = make_uint4(w[0], w[1], w[2], w[3]);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Prep: one unit of 32 x 128 parameter elements per block.  Memory-bound (14 +
// 2 bytes per element); all of a block's loads are issued before its stores.
template <bool NESTEROV>
__global__ __launch_bounds__(256) void direct_prep_kernel(const DirectBatch b, const DirectIndex x, char* ws, float w_mom,
                                                          float w_nest, const float* grad_scale,
                                                          const float* found_inf) {
    constexpr int LD = 128 + 8;  // halves per LDS row (16-byte aligned rows)
    __shared__ __attribute__((aligned(16))) uint16_t tile[32 * LD];
    __shared__ float red[4];
    const int tid = threadIdx.x;
    const int mi = find_matrix(x, blockIdx.x);
    const DirectMat& d = b.d[mi];
    const int unit = int(blockIdx.x) - x.begin[mi];
    if (blockIdx.x == 0 && tid < b.count) reinterpret_cast<DirectMat*>(ws)[tid] = b.d[tid];
    const int R = d.rows, C = d.cols;
    const int pieces = (C + 127) >> 7;  // 128-column pieces per 32-row band
    const int r0 = (unit / pieces) * 32, c0 = (unit % pieces) * 128;
    const int cg = tid & 31, rr = tid >> 5;
    const int c = c0 + cg * 4;
    const bool gb = (d.flags & MAMW_BF16_GRAD) != 0;
    const float* gf = static_cast<const float*>(d.grad);
    const uint16_t* gh = static_cast<const uint16_t*>(d.grad);
    const bool vec = (C & 3) == 0 && (reinterpret_cast<uintptr_t>(d.grad) & (gb ? 7 : 15)) == 0 &&
                     (reinterpret_cast<uintptr_t>(d.mom) & 15) == 0;
    const bool scaled = grad_scale != nullptr;
    const float gsc = scaled ? *grad_scale : 1.0f;
    const bool keep_mom = !(found_inf && *found_inf != 0.0f);
    float g[4][4], m[4][4], u[4][4];
    // Element e of pass p: row r0 + rr + 8 p, column c + e (zero outside).
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const int r = r0 + rr + 8 * p;
        const int64_t off = int64_t(r) * C + c;
#pragma unroll
        for (int e = 0; e < 4; ++e) g[p][e] = m[p][e] = 0.f;
        if (r >= R) continue;
        if (vec) {
            if (c < C) {
                if (gb) {
                    const uint2 w = *reinterpret_cast<const uint2*>(gh + off);
                    g[p][0] = bf16_to_f32(w.x & 0xffffu);
                    g[p][1] = bf16_to_f32(w.x >> 16);
                    g[p][2] = bf16_to_f32(w.y & 0xffffu);
                    g[p][3] = bf16_to_f32(w.y >> 16);
                } else {
                    const f32x4_t v = *reinterpret_cast<const f32x4_t*>(gf + off);
#pragma unroll
                    for (int e = 0; e < 4; ++e) g[p][e] = v[e];
                }
                const f32x4_t v = *reinterpret_cast<const f32x4_t*>(d.mom + off);
#pragma unroll
                for (int e = 0; e < 4; ++e) m[p][e] = v[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (c + e < C) {
                    g[p][e] = gb ? bf16_to_f32(gh[off + e]) : gf[off + e];
                    m[p][e] = d.mom[off + e];
                }
            }
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const int r = r0 + rr + 8 * p;
        const int64_t off = int64_t(r) * C + c;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const bool in = r < R && c + e < C;
            const float gv = scaled ? g[p][e] / gsc : g[p][e];
            m[p][e] = lerp_torch(m[p][e], gv, w_mom);
            u[p][e] = in ? (NESTEROV ? lerp_torch(gv, m[p][e], w_nest) : m[p][e]) : 0.f;
        }
        if (keep_mom && r < R) {
            if (vec) {
                if (c < C) *reinterpret_cast<f32x4_t*>(d.mom + off) = f32x4_t{m[p][0], m[p][1], m[p][2], m[p][3]};
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (c + e < C) d.mom[off + e] = m[p][e];
            }
        }
        const uint2 pk = make_uint2(pack_bf16x2(u[p][0], u[p][1]), pack_bf16x2(u[p][2], u[p][3]));
        const uint32_t h[4] = {pk.x & 0xffffu, pk.x >> 16, pk.y & 0xffffu, pk.y >> 16};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float xb = bf16_to_f32(h[e]);
            ss += xb * xb;
        }
        *reinterpret_cast<uint2*>(&tile[(rr + 8 * p) * LD + cg * 4]) = pk;
    }
    const float sw = wave_sum(ss);
    if ((tid & 63) == 0) red[tid >> 6] = sw;
    __syncthreads();
    char* base = ws + int64_t(d.ws) * 256;
    if (tid == 0)
        reinterpret_cast<float*>(base + direct_off_part(d.mp, d.np))[unit] = (red[0] + red[1]) + (red[2] + red[3]);
    // Parameter rows are rows of `along` (X of a wide matrix, X^T of a tall
    // one) and columns of `across`.  Each is written as 8 blocks of 1 KB.
    const int Rp = d.tall ? d.np : d.mp, Cp = d.tall ? d.mp : d.np;
    uint16_t* xt = reinterpret_cast<uint16_t*>(base);
    uint16_t* xm = reinterpret_cast<uint16_t*>(base + direct_off_x(d.mp, d.np));
    uint16_t* along = d.tall ? xt : xm;
    uint16_t* across = d.tall ? xm : xt;
    if (r0 < Rp) store_unit<LD>(tile, tid, r0, c0, Rp, Cp, along, across);
}

// A row-major bf16 matrix (rows x cols) into fragment-major matrices padded
// with zeros to Rp x Cp: `along` (its rows are rows) and, if not NULL, `across`
// (its columns are rows).  32 x 128 elements per block.
__global__ __launch_bounds__(256) void direct_pack_kernel(const uint16_t* __restrict__ src, int R, int C, int Rp, int Cp,
                                                          uint16_t* __restrict__ along, uint16_t* __restrict__ across) {
    constexpr int LD = 128 + 8;
    __shared__ __attribute__((aligned(16))) uint16_t tile[32 * LD];
    const int tid = threadIdx.x, pieces = (Cp + 127) >> 7;
    const int r0 = (int(blockIdx.x) / pieces) * 32, c0 = (int(blockIdx.x) % pieces) * 128;
    const bool vec = (C & 7) == 0 && (reinterpret_cast<uintptr_t>(src) & 15) == 0;
    if (vec) {  // 8 columns of rows tid / 16 and + 16
        uint4 w[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int r = r0 + (tid >> 4) + 16 * p, c = c0 + (tid & 15) * 8;
            w[p] = r < R && c < C ? *reinterpret_cast<const uint4*>(src + int64_t(r) * C + c) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) *reinterpret_cast<uint4*>(&tile[((tid >> 4) + 16 * p) * LD + (tid & 15) * 8]) = w[p];
    } else {  // single elements, 128 lanes a row
        uint16_t h[16];
#pragma unroll
        for (int p = 0; p < 16; ++p) {
            const int r = r0 + (tid >> 7) + 2 * p, c = c0 + (tid & 127);
            h[p] = r < R && c < C ? src[int64_t(r) * C + c] : uint16_t(0);
        }
#pragma unroll
        for (int p = 0; p < 16; ++p) tile[((tid >> 7) + 2 * p) * LD + (tid & 127)] = h[p];
    }
    __syncthreads();
    store_unit<LD>(tile, tid, r0, c0, Rp, Cp, along, across);
}

// Norm and scale: X and X^T lie one after the other, 8192 elements per block.
// Every block sums the matrix's partials itself, in muon_norm_kernel's order
// (a launch less; at most kDirectMaxUnits of them, a few loads per thread),
// while its own 64 bytes per thread are on the way.
__global__ __launch_bounds__(256) void direct_scale_kernel(const DirectIndex ix, char* ws, float eps) {
    __shared__ float red[4];
    const int tid = threadIdx.x;
    const int mi = find_matrix(ix, blockIdx.x);
    const DirectMat d = table_entry(ws, mi);
    char* base = ws + int64_t(d.ws) * 256;
    uint4* x = reinterpret_cast<uint4*>(base) + int64_t(int(blockIdx.x) - ix.begin[mi]) * 1024 + tid;
    uint4 w[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) w[p] = x[256 * p];
    const float* part = reinterpret_cast<const float*>(base + direct_off_part(d.mp, d.np));
    const int P = direct_units(d.rows, d.cols);
    float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    int i = tid;
    for (; i + 7 * 256 < P; i += 8 * 256) {
#pragma unroll
        for (int u = 0; u < 8; ++u) a[u] += part[i + u * 256];
    }
    for (; i < P; i += 256) a[0] += part[i];
    float s = ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
    s = wave_sum(s);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    const float tot = (red[0] + red[1]) + (red[2] + red[3]);
    const float nrm = bf16_to_f32(f32_to_bf16(sqrtf(tot)));
    const float inv = 1.0f / bf16_to_f32(f32_to_bf16(fmaxf(nrm, eps)));
#pragma unroll
    for (int p = 0; p < 4; ++p) x[256 * p] = scale_bf16x8(w[p], inv);
}

// ---------------------------------------------------------------------------
// One wavefront computes the T x T tile C[y][x] = sum_k Yop[y][k] * Xop[x][k].
// Gram and polynomial: y = i, x = j, tiles with y <= x, written to both
// triangles.  Update: y = i, x = j (Yop = B, Xop = X^T).  Apply: x runs along
// the parameter's columns, so that 32 lanes touch one parameter row: y = i for
// a wide matrix, y = j (Yop = X^T, Xop = B) for a tall one; the products and
// their order are the same either way.
//
// D - 1 panels of 64 k are in flight (T = 32: 3 of 8 KB; T = 64: 1 of 16 KB);
// past the end of the reduction the last panel is loaded again and not used.
struct DirectGemm {
    // Equal-shaped matrices (tiles > 0): every block's matrix and addresses
    // follow from these, without a read of the launch table that depends on
    // another (each such read is a memory latency of about 0.6 us).
    int mp, np, tiles;
    uint32_t stride;  // workspace bytes of a matrix / 256
    int total;        // launch blocks
    float alpha;  // coefficient on the accumulator (polynomial)
    float beta;   // coefficient on A (polynomial) or X (update, apply)
    float keep;   // apply: 1 - lr * weight_decay
    int cur;      // which X^T buffer holds the iterate
    int super;    // tiles per edge of the square whose tiles are consecutive
    const float* found_inf;
    uint16_t* out;  // ROWMAJOR: output, its rows and columns
    int orows, ocols;
};

// ROWMAJOR: the product goes out as a row-major bf16 matrix (the standalone
// functions), rows and columns beyond it dropped.
template <int MODE, int T, bool ROWMAJOR = false>
__global__ __launch_bounds__(64, 2) void direct_gemm_kernel(char* ws, const DirectGemm g, const DirectIndex ix) {
    constexpr bool SYM = MODE == DM_GRAM || MODE == DM_POLY;
    constexpr int F = T / 32;              // fragments per tile edge
    constexpr int D = T == 32 ? 4 : 2;     // panels of 64 k in the register ring
    // Halves per LDS row of a 32 x 32 fragment; rows read as 16-byte chunks are aligned.
    constexpr int LD = ROWMAJOR ? 40 : 36;
    __shared__ __attribute__((aligned(16))) uint16_t tr[32 * LD];
    if constexpr (MODE == DM_APPLY) {
        if (g.found_inf && *g.found_inf != 0.0f) return;
    }
    const int lane = threadIdx.x;
    // All scalar arguments in one read (the compiler would fetch them where
    // they are first used, each a latency of its own: 1 us of a 50 us step).
    asm volatile("" ::"s"(g.mp), "s"(g.np), "s"(g.tiles), "s"(g.stride), "s"(g.cur), "s"(g.super), "s"(g.total), "s"(ws),
                 "s"(g.alpha), "s"(g.beta));
    const int block = xcd_contiguous(blockIdx.x, g.total);
    int mi, t, ty, tx, mp = g.mp, np = g.np;
    uint32_t region;
    if (g.tiles > 0) {
        mi = __builtin_amdgcn_readfirstlane(block / g.tiles);
        t = block - mi * g.tiles;
        region = uint32_t(kDirectTableBytes / 256) + uint32_t(mi) * g.stride;
    } else {
        mi = find_matrix(ix, block);
        t = block - ix.begin[mi];
    }
    const DirectMat d = table_entry(ws, mi);
    if (g.tiles <= 0) {
        mp = d.mp;
        np = d.np;
        region = d.ws;
    }
    if constexpr (SYM) {
        // Super column J of w tile columns: J squares of super x w tiles, then
        // the triangle on the diagonal.
        const int S = g.super, n = mp / T;
        int J = 0, w = min(S, n);
        for (;;) {
            const int tiles = J * S * w + w * (w + 1) / 2;
            if (t < tiles) break;
            t -= tiles;
            ++J;
            w = min(S, n - J * S);
        }
        if (t < J * S * w) {
            ty = (t / (S * w)) * S + t % S;
            tx = J * S + (t % (S * w)) / S;
        } else {
            t -= J * S * w;
            int c = 0;
            while (t > c) t -= ++c;
            ty = J * S + t;
            tx = J * S + c;
        }
    } else {
        // Super columns (along n) of w tile columns, each walked by squares.
        const int S = g.super, rows = mp / T, cols = np / T;
        const int J = t / (rows * S), w = min(S, cols - J * S);
        t -= J * rows * S;
        const int I = t / (S * w), h = min(S, rows - I * S);
        t -= I * S * w;
        ty = I * S + t % h;
        tx = J * S + t / h;
    }
    const bool swap = MODE == DM_APPLY && d.tall;
    if (swap) {
        const int s = ty;
        ty = tx;
        tx = s;
    }
    ty = __builtin_amdgcn_readfirstlane(ty);
    tx = __builtin_amdgcn_readfirstlane(tx);

    char* base = ws + int64_t(region) * 256;
    uint16_t* const X = reinterpret_cast<uint16_t*>(base + direct_off_x(mp, np));
    uint16_t* const XT = reinterpret_cast<uint16_t*>(base + (g.cur ? direct_off_xt1(mp, np) : 0));
    uint16_t* const A = reinterpret_cast<uint16_t*>(base + direct_off_a(mp, np));
    uint16_t* const B = reinterpret_cast<uint16_t*>(base + direct_off_b(mp, np));
    const uint16_t* yop = MODE == DM_GRAM ? X : MODE == DM_POLY ? A : swap ? XT : B;
    const uint16_t* xop = MODE == DM_GRAM ? X : MODE == DM_POLY ? A : swap ? B : XT;
    const int yrows = SYM || !swap ? mp : np, xrows = SYM || swap ? mp : np;
    const int K = MODE == DM_GRAM ? np : mp, P = K >> 6;

    // Epilogue coefficient, 4 consecutive y of one x per group: A (symmetric),
    // or X as X^T (rows j) or as X (rows i, swapped).
    uint2 coef[F][F][4];
    if constexpr (MODE != DM_GRAM) {
        const uint16_t* src = MODE == DM_POLY ? A : swap ? X : XT;
#pragma unroll
        for (int a = 0; a < F; ++a)
#pragma unroll
            for (int c = 0; c < F; ++c)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    coef[a][c][q] = *reinterpret_cast<const uint2*>(
                        src + foff(xrows, tx * T + c * 32 + (lane & 31), ty * T + a * 32 + q * 8 + (lane >> 5) * 4));
    }

    // Apply: a tile that lies inside the parameter loads its elements now, so
    // that their HBM latency passes under the operands'.
    // Lane: column x = tx T + 32 c + lane % 32, rows 4 (lane / 32) + constants,
    // whose offsets ride in the scalar offset.
    const bool bf = MODE == DM_APPLY && (d.flags & MAMW_BF16_PARAM) != 0;
    const int R = MODE == DM_APPLY ? d.rows : 0, C = MODE == DM_APPLY ? d.cols : 0;
    const bool inner = MODE == DM_APPLY && (tx + 1) * T <= C && (ty + 1) * T <= R;
    const int es = bf ? 2 : 4;
    const __amdgpu_buffer_rsrc_t rp = rsrc(MODE == DM_APPLY ? d.param : nullptr, int64_t(R) * C * es);
    const __amdgpu_buffer_rsrc_t ru = rsrc(MODE == DM_APPLY ? d.upd : nullptr, MODE == DM_APPLY && d.upd ? int64_t(R) * C * 4 : 0);
    const int at0 = (ty * T + (lane >> 5) * 4) * C + tx * T + (lane & 31);
    uint32_t pre[F][F][16];
    if constexpr (MODE == DM_APPLY) {
        if (inner) {
#pragma unroll
            for (int a = 0; a < F; ++a)
#pragma unroll
                for (int c = 0; c < F; ++c)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int so = (a * 32 + (e >> 2) * 8 + (e & 3)) * C + c * 32;
                        pre[a][c][e] = bf ? uint32_t(__builtin_amdgcn_raw_buffer_load_b16(rp, at0 * 2, so * 2, 0))
                                          : __builtin_amdgcn_raw_buffer_load_b32(rp, at0 * 4, so * 4, 0);
                    }
        }
    }

    const __amdgpu_buffer_rsrc_t ry = rsrc(yop, int64_t(yrows) * K * 2), rx = rsrc(xop, int64_t(xrows) * K * 2);
    const int vo = lane * 16, py = yrows * 32, px = xrows * 32;  // bytes of one 16-wide column of blocks
    f32x16_t acc[F][F];
#pragma unroll
    for (int a = 0; a < F; ++a)
#pragma unroll
        for (int c = 0; c < F; ++c)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[a][c][e] = 0.f;
    u32x4_t fy[D][4][F], fx[D][4][F];
    auto load = [&](int s, int p) __attribute__((always_inline)) {
        p = min(p, P - 1);
        const int sy = 4 * p * py + ty * T * 32, sx = 4 * p * px + tx * T * 32;
#pragma unroll
        for (int h = 0; h < 4; ++h) {
#pragma unroll
            for (int a = 0; a < F; ++a) fy[s][h][a] = __builtin_amdgcn_raw_buffer_load_b128(ry, vo, sy + h * py + a * 1024, 0);
#pragma unroll
            for (int c = 0; c < F; ++c) fx[s][h][c] = __builtin_amdgcn_raw_buffer_load_b128(rx, vo, sx + h * px + c * 1024, 0);
        }
    };
    auto mma = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 4; ++h)
#pragma unroll
            for (int a = 0; a < F; ++a)
#pragma unroll
                for (int c = 0; c < F; ++c)
                    acc[a][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, fy[s][h][a]),
                                                                        __builtin_bit_cast(bf16x8_t, fx[s][h][c]),
                                                                        acc[a][c], 0, 0, 0);
    };
#pragma unroll
    for (int s = 0; s < D - 1; ++s) load(s, s);
    int p = 0;
    for (; p + D <= P; p += D) {
#pragma unroll
        for (int s = 0; s < D; ++s) {
            load((s + D - 1) % D, p + s + D - 1);
            mma(s);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int s = 0; s < D - 1; ++s)
        if (p + s < P) mma(s);

    // Lane holds, for fragment (a, c) and group q, C[y .. y+3][x] with
    // x = tx T + 32 c + lane % 32, y = ty T + 32 a + 8 q + 4 (lane / 32).
    auto value = [&](int a, int c, int q) __attribute__((always_inline)) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[a][c][q * 4 + e];
        if constexpr (MODE != DM_GRAM) {
            const uint2 s2 = coef[a][c][q];
            const float sv[4] = {bf16_to_f32(s2.x & 0xffffu), bf16_to_f32(s2.x >> 16), bf16_to_f32(s2.y & 0xffffu),
                                 bf16_to_f32(s2.y >> 16)};
#pragma unroll
            for (int e = 0; e < 4; ++e)
                v[e] = MODE == DM_POLY ? __builtin_fmaf(g.alpha, v[e], g.beta * sv[e]) : __builtin_fmaf(g.beta, sv[e], v[e]);
        }
        return make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
    };

    if constexpr (MODE == DM_APPLY) {
        // 32 lanes of a group read and write 32 consecutive elements of a
        // parameter row; what lies outside the parameter is not touched.
        if (inner) {
#pragma unroll
            for (int a = 0; a < F; ++a)
#pragma unroll
                for (int c = 0; c < F; ++c)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint2 w = value(a, c, q);
                        const float u[4] = {bf16_to_f32(w.x & 0xffffu), bf16_to_f32(w.x >> 16),
                                            bf16_to_f32(w.y & 0xffffu), bf16_to_f32(w.y >> 16)};
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const uint32_t p0 = pre[a][c][q * 4 + e];
                            const float pv = bf ? bf16_to_f32(p0) : __uint_as_float(p0);
                            const float o = __builtin_fmaf(-d.slr, u[e], pv * g.keep);
                            const int so = (a * 32 + q * 8 + e) * C + c * 32;
                            if (bf)
                                __builtin_amdgcn_raw_buffer_store_b16(short(f32_to_bf16(o)), rp, at0 * 2, so * 2, kStoreThrough);
                            else
                                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o), rp, at0 * 4, so * 4, kStoreThrough);
                            if (d.upd) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(u[e]), ru, at0 * 4, so * 4, 0);
                        }
                    }
            return;
        }
#pragma unroll
        for (int a = 0; a < F; ++a)
#pragma unroll
            for (int c = 0; c < F; ++c) {
                const int x = tx * T + c * 32 + (lane & 31), y0 = ty * T + a * 32 + (lane >> 5) * 4;
                int idx[16];
                float pv[16];
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int y = y0 + (e >> 2) * 8 + (e & 3);
                    idx[e] = (x < C && y < R) ? y * C + x : 0x1fffffff;  // beyond both resources
                    pv[e] = bf ? bf16_to_f32(__builtin_amdgcn_raw_buffer_load_b16(rp, idx[e] * 2, 0, 0))
                               : __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rp, idx[e] * 4, 0, 0));
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint2 w = value(a, c, q);
                    const float u[4] = {bf16_to_f32(w.x & 0xffffu), bf16_to_f32(w.x >> 16), bf16_to_f32(w.y & 0xffffu),
                                        bf16_to_f32(w.y >> 16)};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float o = __builtin_fmaf(-d.slr, u[e], pv[q * 4 + e] * g.keep);
                        const int at = idx[q * 4 + e];
                        if (bf)
                            __builtin_amdgcn_raw_buffer_store_b16(short(f32_to_bf16(o)), rp, at * 2, 0, 0);
                        else
                            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o), rp, at * 4, 0, 0);
                        if (d.upd) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(u[e]), ru, at * 4, 0, 0);
                    }
                }
            }
        return;
    }

    if constexpr (ROWMAJOR) {
        // Each fragment through LDS (tr[x][y]), then rows of 64 bytes: 4 lanes
        // a row in 16-byte chunks where the rows allow it, else 32 lanes a row
        // in single elements.
        uint16_t* const out = g.out;
        const int orows = g.orows, ocols = g.ocols;
        const bool vec = (ocols & 7) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
#pragma unroll
        for (int a = 0; a < F; ++a)
#pragma unroll
            for (int c = 0; c < F; ++c) {
                if (SYM && a > c && ty == tx) continue;  // the mirror of (c, a)
                const int x0 = tx * T + c * 32, y0 = ty * T + a * 32;
                if (a + c > 0) __syncthreads();  // the previous fragment has been read
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<uint2*>(&tr[(lane & 31) * LD + q * 8 + (lane >> 5) * 4]) = value(a, c, q);
                __syncthreads();
                // C[y][x]: tr[x][y], of a symmetric product's diagonal fragment
                // the upper triangle (y <= x) for both.
                const bool diag = SYM && x0 == y0;
                auto at = [&](int y, int x) { return diag && y > x ? tr[y * LD + x] : tr[x * LD + y]; };
                const bool mirror = SYM && !diag;
                if (vec) {
                    const int ch = (lane & 3) * 8;
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        const int r = k * 16 + (lane >> 2);
                        uint32_t w[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            w[e] = uint32_t(at(r, ch + 2 * e)) | (uint32_t(at(r, ch + 2 * e + 1)) << 16);
                        if (y0 + r < orows && x0 + ch < ocols)
                            *reinterpret_cast<uint4*>(out + int64_t(y0 + r) * ocols + x0 + ch) = make_uint4(w[0], w[1], w[2], w[3]);
                        if (mirror && x0 + r < orows && y0 + ch < ocols)
                            *reinterpret_cast<uint4*>(out + int64_t(x0 + r) * ocols + y0 + ch) =
                                *reinterpret_cast<const uint4*>(&tr[r * LD + ch]);
                    }
                } else {
                    const int e = lane & 31;
#pragma unroll
                    for (int k = 0; k < 16; ++k) {
                        const int r = 2 * k + (lane >> 5);
                        if (y0 + r < orows && x0 + e < ocols) out[int64_t(y0 + r) * ocols + x0 + e] = at(r, e);
                        if (mirror && x0 + r < orows && y0 + e < ocols) out[int64_t(x0 + r) * ocols + y0 + e] = tr[r * LD + e];
                    }
                }
            }
        return;
    }

    // "Across" (rows x, 4 consecutive y per lane) needs no transpose: lanes l
    // and l + 32 fill one 16-byte chunk.  "Along" (rows y) goes through LDS,
    // one fragment at a time, and comes back by transpose reads: in a 16-lane
    // group lane j names tr[xc + j/4][yb + 4 (j%4) ..], lane i receives
    // C[yb + i][xc .. xc+3].
    uint16_t* const across = MODE == DM_GRAM ? A : MODE == DM_POLY ? B
                           : reinterpret_cast<uint16_t*>(base + (g.cur ? 0 : direct_off_xt1(mp, np)));
    uint16_t* const along = MODE == DM_GRAM ? A : MODE == DM_POLY ? B : X;
    // Stores write through the L2 (kStoreThrough): the tiles of a small launch
    // end together, and what is still dirty in the L2s is written back before
    // the next launch may begin (steps without -> with: two 512 x 2048 113 ->
    // 108 us, four 768 x 768 159 -> 152, 2048 x 2048 319 -> 308).
    const __amdgpu_buffer_rsrc_t r_across = rsrc(across, int64_t(xrows) * (SYM ? mp : yrows) * 2);
    const __amdgpu_buffer_rsrc_t r_along = rsrc(along, int64_t(yrows) * (SYM ? mp : xrows) * 2);
#pragma unroll
    for (int a = 0; a < F; ++a)
#pragma unroll
        for (int c = 0; c < F; ++c) {
            if (SYM && a > c && ty == tx) continue;  // the mirror of (c, a)
            const int x0 = tx * T + c * 32, y0 = ty * T + a * 32;
            const bool both = !SYM || x0 != y0;  // a diagonal fragment is its own mirror
            if (both && a + c > 0) __syncthreads();  // the previous fragment has been read
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint2 w = value(a, c, q);
                __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{w.x, w.y}, r_across,
                                                      foff(xrows, x0 + (lane & 31), y0 + q * 8 + (lane >> 5) * 4) * 2, 0,
                                                      kStoreThrough);
                *reinterpret_cast<uint2*>(&tr[(lane & 31) * LD + q * 8 + (lane >> 5) * 4]) = w;
            }
            if (!both) continue;
            __syncthreads();
            const int j = lane & 15, band = (lane >> 4) & 1, half = lane >> 5;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int xc = k * 16 + half * 8;
                const uint16_t* s0 = &tr[(xc + (j >> 2)) * LD + band * 16 + 4 * (j & 3)];
                const uint2 lo = __builtin_bit_cast(
                    uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_ptr_t)(lds_ptr_t)(const_cast<uint16_t*>(s0))));
                const uint2 hi = __builtin_bit_cast(
                    uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_ptr_t)(lds_ptr_t)(const_cast<uint16_t*>(s0 + 4 * LD))));
                __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{lo.x, lo.y, hi.x, hi.y}, r_along,
                                                       foff(yrows, y0 + band * 16 + j, x0 + xc) * 2, 0, kStoreThrough);
            }
        }
}

// Tiles of a product over the launch's matrices.
template <int MODE>
int64_t count_tiles(const DirectBatch& b, int T) {
    int64_t total = 0;
    for (int i = 0; i < b.count; ++i) {
        const int64_t r = b.d[i].mp / T, c = b.d[i].np / T;
        total += (MODE == DM_GRAM || MODE == DM_POLY) ? r * (r + 1) / 2 : r * c;
    }
    return total;
}

// 64-wide tiles move half the operand bytes per flop, 32-wide ones spread a
// small product over four times the CUs: 64 from 1.5 tiles per CU on.  Whole
// steps, 32 against 64 on the symmetric products: 1024 x 4096 (136 64-wide
// tiles) 198 / 297 us, 4 x 768 x 3072 (312) 332 / 344, 8 x 512 x 512 (288)
// 118 / 118, 2048 x 2048 (528) 400 / 320; on the updates: 4 x 256 x 1024 (256)
// 78 / 84, 2 x 512 x 2048 (512) 122 / 119, 768 x 3072 (576) 157 / 151.
constexpr int64_t kDirectWideTiles = 384;

template <int MODE, bool ROWMAJOR = false>
hipError_t launch_direct(const DirectBatch& b, char* ws, const DirectGemm& g, double flops, hipStream_t s) {
    const int T = count_tiles<MODE>(b, 64) >= kDirectWideTiles ? 64 : 32;
    DirectIndex x{};
    x.count = b.count;
    int64_t total = 0;
    int m = 0;
    for (int i = 0; i < b.count; ++i) {
        x.begin[i] = int32_t(total);
        const int64_t r = b.d[i].mp / T, c = b.d[i].np / T;
        total += (MODE == DM_GRAM || MODE == DM_POLY) ? r * (r + 1) / 2 : r * c;
        const int mi = b.d[i].tall ? b.d[i].cols : b.d[i].rows;
        m = m > mi ? m : mi;
    }
    constexpr int32_t kid = MODE == DM_GRAM ? K_DIRECT_GRAM : MODE == DM_POLY ? K_DIRECT_POLY
                          : MODE == DM_UPDATE ? K_DIRECT_UPDATE : K_DIRECT_APPLY;
    DirectGemm ga = g;
    // Consecutive blocks cover squares of 128, in the updates of matrices with
    // m >= 1024 of 256 (the tiles the staged kernels use there).
    const int square = (MODE == DM_UPDATE || MODE == DM_APPLY) && m >= 1024 ? 256 : 128;
    ga.super = square / T;
    ga.total = int(total);
    if (b.uniform) {
        ga.mp = b.d[0].mp;
        ga.np = b.d[0].np;
        ga.tiles = int(total / b.count);
        ga.stride = b.count > 1 ? b.d[1].ws - b.d[0].ws : 0;
    }
    const dim3 grid{unsigned(total)}, block{64};
    if (T == 64) return launch(kid, 8 * square, flops, 0.0, direct_gemm_kernel<MODE, 64, ROWMAJOR>, grid, block, s, ws, ga, x);
    return launch(kid, 8 * square, flops, 0.0, direct_gemm_kernel<MODE, 32, ROWMAJOR>, grid, block, s, ws, ga, x);
}

}  // namespace
}  // namespace mamw

using namespace mamw;

extern "C" int mamw_muon_direct_workspace_bytes(const mamw_muon_matrix* mats, int count, int ns_steps, size_t* bytes) {
    if (!bytes || !mats) return MAMW_ERR_NULL;
    return direct_workspace(mats, count, ns_steps, bytes);
}

extern "C" int mamw_muon_direct_step(const mamw_muon_matrix* mats, int count, double lr, double weight_decay,
                                     double beta, int nesterov, float a, float b, float c, int ns_steps, float eps,
                                     void* workspace, size_t workspace_bytes, const float* grad_scale,
                                     const float* found_inf, mamw_stream_t stream) {
    DirectBatch B;
    const int st = direct_validate(mats, count, ns_steps, workspace, workspace_bytes, &B);
    if (st != MAMW_OK) return st;
    hipStream_t s = static_cast<hipStream_t>(stream);
    char* ws = static_cast<char*>(workspace);
    double elems = 0.0, f_gram = 0.0, f_poly = 0.0, f_upd = 0.0, padded = 0.0;
    for (int i = 0; i < count; ++i) {
        const DirectMat& d = B.d[i];
        const double m = d.tall ? d.cols : d.rows, n = d.tall ? d.rows : d.cols;
        elems += m * n;
        padded += double(d.mp) * d.np;
        f_gram += m * m * n;
        f_poly += m * m * m;
        f_upd += 2.0 * m * m * n;
    }
    DirectIndex x{};
    x.count = count;
    int64_t blocks = 0;
    for (int i = 0; i < count; ++i) {
        x.begin[i] = int32_t(blocks);
        blocks += direct_units(B.d[i].rows, B.d[i].cols);
    }
    const float w_mom = float(1.0 - beta), w_nest = float(beta);
    hipError_t e = nesterov ? launch(K_DIRECT_PREP, 1, 0.0, 16.0 * elems, direct_prep_kernel<true>, dim3(unsigned(blocks)),
                                     dim3(256), s, B, x, ws, w_mom, w_nest, grad_scale, found_inf)
                            : launch(K_DIRECT_PREP, 0, 0.0, 16.0 * elems, direct_prep_kernel<false>, dim3(unsigned(blocks)),
                                     dim3(256), s, B, x, ws, w_mom, w_nest, grad_scale, found_inf);
    if (e != hipSuccess) return int(e);
    blocks = 0;
    for (int i = 0; i < count; ++i) {
        x.begin[i] = int32_t(blocks);
        blocks += int64_t(B.d[i].mp) * B.d[i].np / 4096;
    }
    e = launch(K_DIRECT_SCALE, 0, 0.0, 8.0 * padded, direct_scale_kernel, dim3(unsigned(blocks)), dim3(256), s, x, ws, eps);
    if (e != hipSuccess) return int(e);
    DirectGemm g{};
    g.keep = float(1.0 - lr * weight_decay);
    g.found_inf = found_inf;
    for (int it = 0; it < ns_steps; ++it) {
        g.cur = it & 1;
        e = launch_direct<DM_GRAM>(B, ws, g, f_gram, s);
        if (e != hipSuccess) return int(e);
        g.alpha = c;
        g.beta = b;
        e = launch_direct<DM_POLY>(B, ws, g, f_poly, s);
        if (e != hipSuccess) return int(e);
        g.beta = a;
        e = it == ns_steps - 1 ? launch_direct<DM_APPLY>(B, ws, g, f_upd, s)
                               : launch_direct<DM_UPDATE>(B, ws, g, f_upd, s);
        if (e != hipSuccess) return int(e);
    }
    return MAMW_OK;
}

// ---------------------------------------------------------------------------
// Standalone products of one row-major matrix.

extern "C" int mamw_ns_direct_workspace_bytes(int64_t m, int64_t n, size_t* bytes) {
    if (!bytes) return MAMW_ERR_NULL;
    DirectMat d;
    return ns_direct_plan(m, n, &d, bytes);
}

extern "C" int mamw_ns_direct(int op, const uint16_t* X, const uint16_t* S, uint16_t* out, int64_t m, int64_t n, float a,
                              float b, float c, void* workspace, size_t workspace_bytes, mamw_stream_t stream) {
    if (op < MAMW_NS_GRAM || op > MAMW_NS_STEP) return MAMW_ERR_HYPER;
    DirectBatch B{};
    size_t need = 0;
    int st = ns_direct_plan(m, op == MAMW_NS_POLY ? m : n, &B.d[0], &need);
    if (st != MAMW_OK) return st;
    st = ns_direct_validate(op, X, S, out, m, n, workspace, workspace_bytes, need);
    if (st != MAMW_OK) return st;
    B.count = B.uniform = 1;
    hipStream_t s = static_cast<hipStream_t>(stream);
    char* ws = static_cast<char*>(workspace);
    char* base = ws + kDirectTableBytes;
    const int mp = B.d[0].mp, np = B.d[0].np;
    uint16_t* const xt = reinterpret_cast<uint16_t*>(base);
    uint16_t* const x = reinterpret_cast<uint16_t*>(base + direct_off_x(mp, np));
    uint16_t* const A = reinterpret_cast<uint16_t*>(base + direct_off_a(mp, np));
    uint16_t* const Bm = reinterpret_cast<uint16_t*>(base + direct_off_b(mp, np));
    auto pack = [&](const uint16_t* src, int64_t cols, int cp, uint16_t* along, uint16_t* across) {
        return launch(K_DIRECT_PACK, 0, 0.0, double(m) * double(cols) * 2.0 * (1 + (along != nullptr) + (across != nullptr)),
                      direct_pack_kernel, dim3(unsigned(mp / 32) * unsigned((cp + 127) / 128)), dim3(256), s, src, int(m),
                      int(cols), mp, cp, along, across);
    };
    DirectGemm g{};
    g.out = out;
    g.orows = int(m);
    g.ocols = int(op == MAMW_NS_GRAM || op == MAMW_NS_POLY ? m : n);
    const double M = double(m), N = double(n);
    hipError_t e = op == MAMW_NS_POLY ? pack(X, m, mp, A, nullptr)
                                      : pack(X, n, np, op == MAMW_NS_UPDATE ? nullptr : x, op == MAMW_NS_GRAM ? nullptr : xt);
    if (e == hipSuccess && op == MAMW_NS_UPDATE) e = pack(S, m, mp, Bm, nullptr);
    if (e != hipSuccess) return int(e);
    if (op == MAMW_NS_GRAM) return int(launch_direct<DM_GRAM, true>(B, ws, g, M * M * N, s));
    if (op == MAMW_NS_STEP) {
        e = launch_direct<DM_GRAM>(B, ws, g, M * M * N, s);
        if (e != hipSuccess) return int(e);
    }
    g.alpha = c;
    g.beta = b;
    if (op == MAMW_NS_POLY) return int(launch_direct<DM_POLY, true>(B, ws, g, M * M * M, s));
    if (op == MAMW_NS_STEP) {
        e = launch_direct<DM_POLY>(B, ws, g, M * M * M, s);
        if (e != hipSuccess) return int(e);
    }
    g.beta = a;
    return int(launch_direct<DM_UPDATE, true>(B, ws, g, 2.0 * M * M * N, s));
}
