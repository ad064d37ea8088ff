// Internal layouts and kernel interfaces of the radiance cache (rcache.cpp,
// rcache.hip), apart from the frame pipeline's in dn_internal.h. Nothing here
// is part of the public C-ABI.
#pragma once
#include "dn_internal.h"

// Radiance cache network: multiresolution hash encoding (RC_LEVELS levels of
// RC_FEAT features) plus an MLP of four weight matrices (3 hidden layers of
// RC_W with ReLU, linear output of 3), no biases. Weights are stored row-major
// [out][in] and zero-padded: W0 64x48 (38 inputs used), W1 64x64, W2 64x64,
// W3 16x64 (3 outputs used). A sample row is 16 floats: position (voxel
// units) 3, normal 3, albedo 3, target 3, valid (0/1), 3 unused.
enum {
    RC_LEVELS = 16, RC_FEAT = 2, RC_ENC = 32, RC_IN = 48, RC_W = 64, RC_OUT = 16, RC_SAMPLE = 16,
    RC_OFF_W0 = 0, RC_OFF_W1 = 3072, RC_OFF_W2 = 7168, RC_OFF_W3 = 11264, RC_NPARAM = 12288
};

// The bf16 copies of the weights are kept in the order in which the matrix
// instructions take them, so a lane's A operand is one contiguous piece of LDS
// (16 bytes for v_mfma_f32_16x16x32_bf16, 8 for v_mfma_f32_16x16x16_bf16) and
// a wave's 64 pieces are consecutive: a conflict-free read. Position, within a
// matrix of `cols` columns (16, 48 or 64), of element (row, col): 16-row blocks,
// in each its 32-column blocks, then the 16-column block that is left over. In a
// block, lane 16 q + r (r = row mod 16) holds the columns 4 q + 0..3 of the
// block's one or two 16-column halves.
__host__ __device__ inline uint32_t rc_fragment_index(uint32_t cols, uint32_t row, uint32_t col)
{
    const uint32_t c = col & 31u, lane = 16u * ((c & 15u) >> 2) + (row & 15u), j = c & 3u;
    const uint32_t block = (row >> 4) * 16u * cols + (col >> 5) * 512u;
    return (col >> 5) < (cols >> 5) ? block + lane * 8u + (c >> 4) * 4u + j : block + lane * 4u + j;
}

// Matrix that weight i belongs to: its offset, rows and columns.
__host__ __device__ inline void rc_weight_matrix(uint32_t i, uint32_t& off, uint32_t& rows, uint32_t& cols)
{
    if(i < RC_OFF_W1) { off = RC_OFF_W0; rows = 64; cols = 48; }
    else if(i < RC_OFF_W2) { off = RC_OFF_W1; rows = 64; cols = 64; }
    else if(i < RC_OFF_W3) { off = RC_OFF_W2; rows = 64; cols = 64; }
    else { off = RC_OFF_W3; rows = 16; cols = 64; }
}

// Positions of weight i of the row-major layout in the fragment order of its
// matrix (forward) and of the matrix's transpose (backward).
__host__ __device__ inline void rc_fragment_positions(uint32_t i, uint32_t& forward, uint32_t& transposed)
{
    uint32_t off, rows, cols;
    rc_weight_matrix(i, off, rows, cols);
    const uint32_t r = (i - off) / cols, c = (i - off) % cols;
    forward = off + rc_fragment_index(cols, r, c);
    transposed = off + rc_fragment_index(rows, c, r);
}

struct DNrcNet {
    uint32_t log2T;
    uint32_t denseMask;            // bit l: level l indexes densely ((N_l + 2)^3 <= T)
    uint32_t res[RC_LEVELS];       // N_l
    float extent;                  // positions / extent in [0, 1)
    uint32_t* tab16;               // [L][T] two bf16 features per entry
    float* tab32;                  // [L][T][2] master copy
    float* tabGrad;
    float* tabM;
    float* tabV;
    uint16_t* w16;                 // [RC_NPARAM] bf16 in fragment order
    uint16_t* wT16;                // the transposed matrices in fragment order, for backward
    float* w32;                    // master copy
    float* wGrad;
    float* wM;
    float* wV;
    // Exponential moving average of the parameters over the Adam steps, and
    // its debiased bf16 copies, which predictions use.
    float* tabE;
    uint32_t* tabE16;
    float* wE;
    uint16_t* wE16;
};
// Per-batch buffers of training.
struct DNrcActs {
    uint32_t* x0;                  // [RC_LEVELS][samples] a level's two bf16 features
    float* denc;                   // [RC_LEVELS][samples][2] gradients of the encoded features
    // Table gradients by bucket (rc_bucketed): positions over the extent, the
    // records of every level, bucket and sorting block, those of every level and
    // bucket, and per level 8 * samples record words in bucket order (16 * sample
    // + which of its four corner rows meet the bucket).
    float* unit;                   // [samples][4]
    uint32_t* blockCount;          // [RC_LEVELS][RC_SORT_BLOCKS][RC_MAX_BUCKETS]
    uint32_t* bucketCount;         // [RC_LEVELS][RC_MAX_BUCKETS]
    uint32_t* records;
};
// A bucket: 2^12 consecutive table entries, whose gradients fill 64 KiB of LDS.
enum { RC_BUCKET_LOG2 = 12, RC_MAX_BUCKETS = 128, RC_SORT_BLOCKS = 64, RC_BUCKETED_MAX = 1 << 24 };
// Whether a step on n samples sorts its table gradients by bucket (n up to RC_BUCKETED_MAX).
bool rc_bucketed(const DNrcNet& net, uint32_t n);
struct DNrcAdam {
    float lr, beta1, beta2, eps;
    float bias1, bias2;            // 1 - beta^t
    float emaDecay;                // d: E = d * E + (1 - d) * W after each step
    float emaScale;                // 1 / (1 - d^t): debiasing of E (which starts at 0)
};

// pred: float4 per row (3 outputs plus the row's exact term, the row's valid flag).
int dn_rc_predict(const DNrcNet& net, const float* samples, uint32_t n, float* pred, hipStream_t stream);
// A second stream for training: the corner rows are sorted on it beside the encoding
// and the MLP (`fork` and `join` order it after what came before and before the table
// gradients).
struct DNrcSide {
    hipStream_t stream;
    hipEvent_t fork, join;
};
// side: null runs every kernel on `stream`.
int dn_rc_train(const DNrcNet& net, const float* samples, uint32_t n, const DNrcActs& a, hipStream_t stream,
                const DNrcSide* side = nullptr);
int dn_rc_adam(const DNrcNet& net, const DNrcAdam& opt, hipStream_t stream);
// `batches` batches of n training samples, batch k drawn with seed + k * seedStride
int dn_rc_samples(const DNlightParams& p, uint32_t maxRequests, uint32_t n, uint32_t batches, uint32_t seed,
                  uint32_t seedStride, float* samples, hipStream_t stream);
int dn_rc_gather(const DNlightParams& p, uint32_t slots, float* samples, hipStream_t stream);
int dn_accumulate_f64(const float* src, double* dst, size_t n, hipStream_t stream);
// acc[slot] (4 doubles: rgb sum, count) += samplesPerVoxel (rounded up to the
// work split) independent samples of every stored voxel of the request list.
int dn_rc_reference(const DNlightParams& p, uint32_t slots, uint32_t samplesPerVoxel, uint32_t seed, double* acc,
                    hipStream_t stream);
