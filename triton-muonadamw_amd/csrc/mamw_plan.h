// Host-side planning and validation for the MuonAdamW kernels.
//
// Pure C++ (no HIP headers): everything here runs on the host before any HIP
// call, so argument errors surface as negative status codes on machines
// without a GPU as well.  The device records defined here are shared with the
// kernels (they include this header).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "muonadamw_amd.h"

namespace mamw {

// ---------------------------------------------------------------------------
// AdamW multi-tensor table.
//
// Device layout: n_tensors AdamWRec records (64 bytes each).  Launch block b
// belongs to the tensor t with rec[t].block_begin <= b < rec[t+1].block_begin
// (the block count closes the last range), and covers elements
// [(b - block_begin) * kAdamWChunk, +kAdamWChunk) of that tensor.
constexpr int kAdamWThreads = 256;
constexpr int kAdamWUnroll = 1;  // float4 groups per thread per block
constexpr int64_t kAdamWChunk = int64_t(kAdamWThreads) * 4 * kAdamWUnroll;  // 1024

struct alignas(16) AdamWRec {
    void* p;         // fp32, or bf16 with MAMW_BF16_PARAM
    const void* g;   // fp32, or bf16 with MAMW_BF16_GRAD
    float* m;
    float* v;
    int64_t numel;
    int64_t block_begin;
    int32_t vec_ok;  // every base pointer aligned for 4-element vector access
    int32_t flags;   // MAMW_BF16_* bits
    int32_t pad[2];
};
static_assert(sizeof(AdamWRec) == 64, "AdamWRec must stay 64 bytes");

struct AdamWScalars {
    float lr, bias1, bias2, beta1, beta2, weight_decay, eps;
};

int adamw_validate_tensor(const mamw_adamw_tensor_ex& t);
int adamw_table_bytes(int n_tensors, size_t* bytes);
int adamw_table_pack(const mamw_adamw_tensor* tensors, int n_tensors,
                     void* host_table, size_t table_bytes, int64_t* n_blocks);
int adamw_table_pack_ex(const mamw_adamw_tensor_ex* tensors, int n_tensors,
                        void* host_table, size_t table_bytes, int64_t* n_blocks);

// ---------------------------------------------------------------------------
// Muon batch plan.
//
// A batch holds matrices that share m = min(rows, cols) and n = max(rows, cols).
// Iterates live in the caller's workspace as zero-padded bf16 matrices:
//   X   [batch][mp][np]   the Newton-Schulz iterate (m x n), updated in place
//   XT0 [batch][np][mp]   its transpose (operand of B X), ping-pong with XT1
//   XT1 [batch][np][mp]   (only when ns_steps >= 2)
//   A   [batch][mp][mp]   Gram X X^T
//   B   [batch][mp][mp]   b A + c A A
//   part[batch][prep_tiles] fp32 partial sums of squares (one per prep unit)
//   inv [batch]           fp32 1 / max(bf16(||X||_F), eps)
constexpr int kPrepTile = 64;  // a prep unit holds kPrepTile^2 = 32 x 128 parameter elements
constexpr size_t kWsAlign = 256;

struct MuonMatDesc {
    float* param;
    const float* grad;
    float* mom;
    float* upd;  // optional orthogonalised-update output (NULL = skip)
    int64_t rows;
    int64_t cols;
    float slr;
    int32_t tall;   // rows > cols: X = bf16(u)^T
    int32_t flags;  // MAMW_BF16_* bits
};

struct MuonBatchDescs {
    MuonMatDesc d[MAMW_MUON_MAX_BATCH];
};

struct MuonPlan {
    int batch;
    int tile;  // GEMM tile edge (128 or 256); mp, np are multiples of it
    int64_t m, n, mp, np;
    int64_t prep_tiles;  // prep units, (mp/64) * (np/64); the prep kernel takes two per block
    int xkb;             // workspace matrices k-blocked: a whole matrix's byte offsets fit 31 bits
    // X is kept only when !xkb (the row-major Gram reads it); otherwise its
    // region is empty and off_x == off_xt0.
    size_t off_x, off_xt0, off_xt1, off_a, off_b, off_part, off_inv;
    size_t bytes;
};

int choose_tile(int64_t m, int64_t n, int batch);
int muon_plan(int batch, int64_t rows, int64_t cols, int ns_steps, MuonPlan* plan);
int muon_validate(const mamw_muon_matrix* mats, int batch, int ns_steps,
                  const void* workspace, size_t workspace_bytes, MuonPlan* plan,
                  MuonBatchDescs* descs);

// ---------------------------------------------------------------------------
// Direct path (muon_direct.hip): up to MAMW_MUON_DIRECT_MAX matrices of any
// shapes in one set of launches.  The workspace starts with the launch table
// (a DirectMat per matrix, written by the prep kernel for those after it);
// then each matrix has its own region, padded to multiples of 64,
// fragment-major:
//   X^T0 [np][mp], X [mp][np] (adjacent: the scale kernel runs over both),
//   X^T1 [np][mp], A [mp][mp], B [mp][mp], the prep units' sums of squares.
constexpr int kDirectPad = 64;
constexpr int kDirectMaxUnits = 1 << 14;                 // prep units per matrix (each scale block sums them all)
constexpr int64_t kDirectMaxElems = int64_t(1) << 26;    // padded elements per matrix (32-bit buffer offsets)

constexpr int64_t direct_off_x(int64_t mp, int64_t np) { return mp * np * 2; }
constexpr int64_t direct_off_xt1(int64_t mp, int64_t np) { return mp * np * 4; }
constexpr int64_t direct_off_a(int64_t mp, int64_t np) { return mp * np * 6; }
constexpr int64_t direct_off_b(int64_t mp, int64_t np) { return mp * np * 6 + mp * mp * 2; }
constexpr int64_t direct_off_part(int64_t mp, int64_t np) { return mp * np * 6 + mp * mp * 4; }
// Prep units of 32 x 128 elements, counted over the parameter padded to 128 x 128
// as the LDS-staged path counts them: the same sums in the same places.
constexpr int direct_units(int rows, int cols) { return ((rows + 127) / 128 * 4) * ((cols + 127) / 128); }

struct DirectMat {
    void* param;
    const void* grad;
    float* mom;
    float* upd;  // optional orthogonalised-update output (NULL = skip)
    int32_t rows, cols;
    int32_t mp, np;
    uint32_t ws;  // workspace offset of the matrix's region, in units of 256 bytes
    float slr;
    int32_t tall, flags;
};
static_assert(sizeof(DirectMat) == 64, "a launch table entry is one cache half line");

constexpr size_t kDirectTableBytes = sizeof(DirectMat) * MAMW_MUON_DIRECT_MAX;

// First launch block of each matrix.
struct DirectIndex {
    int32_t begin[MAMW_MUON_DIRECT_MAX];
    int32_t count;
};

struct DirectBatch {
    DirectMat d[MAMW_MUON_DIRECT_MAX];
    int32_t count;
    int32_t uniform;  // all matrices have one padded shape
};

int direct_workspace(const mamw_muon_matrix* mats, int count, int ns_steps, size_t* bytes);
int direct_validate(const mamw_muon_matrix* mats, int count, int ns_steps, const void* workspace,
                    size_t workspace_bytes, DirectBatch* batch);

// Standalone products (mamw_ns_direct) of an m x n matrix, m and n in any order:
// the plan of its region, and the buffers.
int ns_direct_plan(int64_t m, int64_t n, DirectMat* d, size_t* bytes);
int ns_direct_validate(int op, const void* X, const void* S, const void* out, int64_t m, int64_t n,
                       const void* workspace, size_t workspace_bytes, size_t need);

// Limits (documented in the ABI through the error codes).
constexpr int64_t kMaxDim = int64_t(1) << 20;        // rows, cols <= 2^20
constexpr int64_t kMaxMatElems = int64_t(1) << 34;   // padded m*n per matrix
constexpr int64_t kMaxNumel = int64_t(1) << 40;      // AdamW elements per tensor
constexpr int kMaxTensors = 1 << 20;

// Byte ranges [a, a+na) and [b, b+nb) overlap (empty ranges never do).
bool ranges_overlap(const void* a, size_t na, const void* b, size_t nb);

inline int64_t round_up(int64_t x, int64_t to) { return (x + to - 1) / to * to; }
inline size_t align_ws(size_t x) { return (x + kWsAlign - 1) / kWsAlign * kWsAlign; }

}  // namespace mamw
