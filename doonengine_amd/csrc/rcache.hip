// Learned radiance cache on gfx950 (no counterpart in the reference).
//
// Encoding: multiresolution hash grid (Mueller et al., "Instant Neural Graphics
// Primitives with a Multiresolution Hash Encoding", 2022, sec. 3): per level l
// the 8 corners of the cell around x * N_l + 0.5, trilinear weights, a dense
// index where (N_l + 2)^3 entries fit the table, else the spatial hash
// (x * 1 ^ y * 2654435761 ^ z * 805459861) mod T.
// Network: 4 weight matrices without biases, ReLU between them; operands in
// bfloat16 on v_mfma_f32_16x16x32_bf16 (v_mfma_f32_16x16x16_bf16 for a
// lone 16-wide K block) with FP32 accumulation. Layers are
// computed transposed (D[feature][sample] = W * X^T), so one layer's 16x16
// accumulator tile is, lane for lane, the next layer's B operand: a lane holds
// sample (lane & 15) and features 4 * (lane >> 4) + 0..3 of a 16-feature block.
// Training: forward, backward and the weight gradients (an MFMA product over
// the samples) in one kernel, hash-table gradients by FP32 atomics or summed in
// LDS by bucket, then Adam (Kingma & Ba 2015, algorithm 1) on FP32 master copies.
#include "dn_light.hpp"
#include "rc_internal.h"
#include "doon/doon.h"

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 hwbf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

// Nearest-even bfloat16: v_cvt_pk_bf16_f32, which agrees with rounding the bits
// in integer arithmetic on every float that is not a NaN (NaNs stay NaNs).
__device__ __forceinline__ uint32_t f2bf2(float lo, float hi)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, hwbf16x2));
}
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __forceinline__ float bf2f(uint32_t h) { return __uint_as_float(h << 16); }

__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// Two consecutive K = 16 steps as one v_mfma_f32_16x16x32_bf16 (gfx950):
// c + A0 B0 + A1 B1. A lane group's 8 k-values of A are its 4 of A0 then its
// 4 of A1, and likewise for B, so A and B pair the same 32 k-values (a
// permutation of the K = 32 block, which leaves the dot product a sum over
// the same terms) and two C-layout tiles feed B without any shuffle.
__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x4 b0, bf16x4 b1, f32x4 c)
{
    const s16x8 b = {b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]};
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ bf16x4 ld_bf16x4(const uint16_t* p)
{
    return __builtin_bit_cast(bf16x4, *reinterpret_cast<const uint2*>(p));
}

// A operands of a matrix in fragment order (rc_fragment_index): `block` is the
// element offset of a 16x32 or 16x16 block.
__device__ __forceinline__ bf16x8 a_frag32(const uint16_t* block, uint32_t lane)
{
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(block + lane * 8u));
}
__device__ __forceinline__ bf16x4 a_frag16(const uint16_t* block, uint32_t lane)
{
    return ld_bf16x4(block + lane * 4u);
}

__device__ __forceinline__ bf16x4 to_bf16(f32x4 c)
{
    return __builtin_bit_cast(bf16x4, make_uint2(f2bf2(c[0], c[1]), f2bf2(c[2], c[3])));
}

__device__ __forceinline__ bf16x4 relu_bf16(f32x4 c)
{
    for(int i = 0; i < 4; i++) c[i] = c[i] > 0.0f ? c[i] : 0.0f;
    return to_bf16(c);
}

// Gradient through ReLU: keep d where the layer output h (bf16) is positive.
__device__ __forceinline__ bf16x4 relu_grad(f32x4 d, bf16x4 h)
{
    for(int i = 0; i < 4; i++) d[i] = h[i] > 0 ? d[i] : 0.0f;     // bits of h: not -0, +0 or negative
    return to_bf16(d);
}

// ---------------------------------------------------------------------------
// encoding

// A position over the extent, clamped to the unit cube.
struct UnitPos { float v[3]; };

__device__ __forceinline__ UnitPos unit_pos(const DNrcNet& net, const float* pos)
{
    UnitPos u;
    for(int a = 0; a < 3; a++) u.v[a] = fminf(fmaxf(pos[a] / net.extent, 0.0f), 1.0f);
    return u;
}

// The cell of a level of resolution N that holds a position: its lower corner
// g and the position's fractions f inside it.
struct LevelCell {
    uint32_t g[3];
    float f[3];
};

__device__ __forceinline__ LevelCell level_cell(uint32_t N, const UnitPos& u)
{
    LevelCell c;
    for(int a = 0; a < 3; a++)
    {
        float s = u.v[a] * (float)N + 0.5f;
        float fl = floorf(s);
        c.g[a] = (uint32_t)fl;
        c.f[a] = s - fl;
    }
    return c;
}

// Corner k (bit 0: x + 1, bit 1: y + 1, bit 2: z + 1) of a cell: its table
// entry (dense index, or the spatial hash) and its trilinear weight.
__device__ __forceinline__ uint32_t corner_index(uint32_t N, bool dense, uint32_t mask, const LevelCell& c, uint32_t k)
{
    const uint32_t S = N + 2u;
    const uint32_t cx = c.g[0] + (k & 1u), cy = c.g[1] + ((k >> 1) & 1u), cz = c.g[2] + ((k >> 2) & 1u);
    const uint32_t i = dense ? cx + cy * S + cz * S * S : (cx * 1u) ^ (cy * 2654435761u) ^ (cz * 805459861u);
    return i & mask;
}

__device__ __forceinline__ float corner_weight(const LevelCell& c, uint32_t k)
{
    return ((k & 1u) ? c.f[0] : 1.0f - c.f[0]) * ((k & 2u) ? c.f[1] : 1.0f - c.f[1]) *
           ((k & 4u) ? c.f[2] : 1.0f - c.f[2]);
}

// Two consecutive table entries, which need not start on 8 bytes.
struct __attribute__((packed, aligned(4))) Pair { uint32_t a, b; };

// A level's two features of a position, as bf16 (first feature in the low half).
// `level` is the entry index at which the level's table starts. KIND: every lane
// of the wave is at a dense level (1), at a hashed one (2), or either (0).
template <int KIND>
__device__ __forceinline__ uint32_t encode_level(const uint32_t* tab, uint32_t level, uint32_t N, bool dense,
                                                 uint32_t mask, const UnitPos& u)
{
    const LevelCell c = level_cell(N, u);
    if(KIND) dense = KIND == 1;
    // Corner (x, y, z): x + y S + z S^2, or x ^ y P ^ z P' mod T. Bound by the number of
    // gathers, so a corner and its x neighbour come with one where they lie side by
    // side: on dense levels always, on hashed ones where x is even (their indices then
    // differ in the last bit only). 10^6 rows at 2^19 entries: 171 us against 178.
    const uint32_t S = N + 2u;
    const uint32_t my = dense ? S : 2654435761u, mz = dense ? S * S : 805459861u;
    const uint32_t y0 = c.g[1] * my, z0 = c.g[2] * mz;
    uint32_t e[8];
    uint32_t at[4];
    Pair p[4];
    #pragma unroll
    for(uint32_t j = 0; j < 4u; j++)
    {
        const uint32_t y = (j & 1u) ? y0 + my : y0, z = (j & 2u) ? z0 + mz : z0;
        at[j] = dense ? c.g[0] + (y + z) : (c.g[0] ^ (y ^ z)) & mask;
        // a 32-bit byte offset (the tables hold at most 2^28 entries)
        p[j] = *reinterpret_cast<const Pair*>(reinterpret_cast<const char*>(tab) +
                                              ((level + (dense ? at[j] : at[j] & ~1u)) << 2));
    }
    const bool apart = !dense && (c.g[0] & 1u);
    uint32_t far[4];
    #pragma unroll
    for(uint32_t j = 0; j < 4u; j++) far[j] = 0u;
    if(apart)
    {
        #pragma unroll
        for(uint32_t j = 0; j < 4u; j++)
        {
            const uint32_t y = (j & 1u) ? y0 + my : y0, z = (j & 2u) ? z0 + mz : z0;
            const uint32_t i = ((c.g[0] + 1u) ^ (y ^ z)) & mask;
            far[j] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(tab) + ((level + i) << 2));
        }
    }
    #pragma unroll
    for(uint32_t j = 0; j < 4u; j++)
    {
        const bool second = !dense && (at[j] & 1u);
        e[2 * j] = second ? p[j].b : p[j].a;
        e[2 * j + 1] = apart ? far[j] : (second ? p[j].a : p[j].b);
    }
    float a0 = 0.0f, a1 = 0.0f;
    #pragma unroll
    for(uint32_t k = 0; k < 8u; k++)
    {
        const float w = corner_weight(c, k);
        a0 += w * bf2f(e[k] & 0xFFFFu);
        a1 += w * bf2f(e[k] >> 16);
    }
    return f2bf2(a0, a1);
}

// Encoding of many rows, one level per wave: a lane takes one sample at levels
// 15 - b and b, b = blockIdx mod 8. Workgroups go to the 8 XCDs in turn, so each
// XCD's 4 MiB L2 serves one fine and one coarse level (2 MiB each at 2^19
// entries) instead of all sixteen, and on the coarse levels neighbouring rows
// of a wave share their entries' lines. Level-major output: 256-byte stores.
__global__ __launch_bounds__(256) void k_rc_encode(DNrcNet net, const float* samples, uint32_t n, uint32_t* x0)
{
    const uint32_t b = blockIdx.x & 7u;
    const uint32_t s = (blockIdx.x >> 3) * 256u + threadIdx.x;
    if(s >= n) return;
    const UnitPos u = unit_pos(net, samples + (size_t)s * RC_SAMPLE);
    const uint32_t mask = (1u << net.log2T) - 1u;
    for(uint32_t i = 0; i < 2u; i++)
    {
        const uint32_t l = i ? b : RC_LEVELS - 1u - b;
        const bool dense = (net.denseMask >> l) & 1u;            // the same for the whole wave
        x0[(size_t)l * n + s] = dense ? encode_level<1>(net.tab16, l << net.log2T, net.res[l], true, mask, u)
                                      : encode_level<2>(net.tab16, l << net.log2T, net.res[l], false, mask, u);
    }
}

// Hash-table gradient of few samples, level-major: the waves running at a time work on one
// level's gradient table (4 MiB at 2^19 entries), finest level first.
// Device-scope FP32 atomics are served per cache line that one instruction
// touches, not per lane (measured on MI355X: 64 lanes on 64 scattered lines
// sustain 20.7 G atomics/s, lane pairs on one 8-byte entry 41 G/s, 16 lanes on
// one 64-byte run about 290 G/s). So four lanes take one sample: lane
// q = 2 xb + f adds feature f at the four corners whose x offset is xb. A
// sample's two x-neighbour corners are adjacent entries on a dense level
// (x + S (y + S z)) and, on a hashed level (x ^ h(y, z)), lie in one aligned
// run of entries unless x + 1 carries past it, so each instruction sends two
// corners and both features of a sample to one line. Per 2^17 training
// samples this takes 185 us, against 378 us with one lane per sample (two
// instructions per corner) and per-wave sums of shared entries on the 8
// coarsest levels; with the four-lane layout such sums only cost time
// (8 levels 275 us, 6 levels 239, 4 levels 223).
__global__ __launch_bounds__(256) void k_rc_table_grad(DNrcNet net, const float* samples, uint32_t n, const float* denc)
{
    const uint32_t g = blockIdx.x * 256u + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63u, w = g >> 6;
    const uint32_t waves = (n + 15u) / 16u;                      // per level
    if(w >= RC_LEVELS * waves) return;
    const uint32_t l = RC_LEVELS - 1u - w / waves;
    const uint32_t s = (w % waves) * 16u + (lane >> 2);
    const uint32_t f = lane & 1u, xb = (lane >> 1) & 1u;
    if(s >= n) return;
    const float d = denc[((size_t)l * n + s) * 2u + f];
    if(d == 0.0f) return;                                       // adding +-0 changes no sum
    float* gt = net.tabGrad + ((size_t)l << net.log2T) * 2u;
    const uint32_t N = net.res[l], mask = (1u << net.log2T) - 1u;
    const bool dense = (net.denseMask >> l) & 1u;
    const LevelCell cell = level_cell(N, unit_pos(net, samples + (size_t)s * RC_SAMPLE));
    for(uint32_t j = 0; j < 4u; j++)
    {
        const uint32_t k = (j << 1) | xb;
        atomicAdd(gt + 2u * corner_index(N, dense, mask, cell, k) + f, corner_weight(cell, k) * d);
    }
}

// Hash-table gradient of many samples, without global atomics on scattered
// entries. Those are performed behind the L2s (giving each level to one XCD
// changed nothing: 521 against 534 us per 2^17 samples of a terrain's surface at
// 2^19 entries), so the table is cut into buckets of 2^12 entries, whose
// gradients a block sums in LDS and adds to the table once. A sample's four
// corner rows (y, z), of two x-neighbour corners each, are first sorted by
// bucket: k_rc_bucket_count, then k_rc_bucket_place, which writes a word per
// sample and bucket that it meets. A level that fits one bucket needs no records.
// The sums are in FP64: LDS atomics on doubles take 22 cycles per wave here, on
// floats 195 whatever the addresses (on 32-bit integers 9).

__device__ __forceinline__ uint32_t level_buckets(const DNrcNet& net, uint32_t l)
{
    const uint32_t S = net.res[l] + 2u, T = 1u << net.log2T;
    const uint32_t entries = ((net.denseMask >> l) & 1u) ? S * S * S : T;
    return (entries + (1u << RC_BUCKET_LOG2) - 1u) >> RC_BUCKET_LOG2;
}

// The buckets that a sample's corners lie in, one of eight values per corner.
struct SampleBuckets {
    uint32_t b[8];
    __device__ __forceinline__ SampleBuckets(uint32_t N, bool dense, uint32_t mask, const UnitPos& u)
    {
        const LevelCell c = level_cell(N, u);
        #pragma unroll
        for(uint32_t k = 0; k < 8u; k++) b[k] = corner_index(N, dense, mask, c, k) >> RC_BUCKET_LOG2;
    }
    // whether corner k is the first one in its bucket
    __device__ __forceinline__ bool first(uint32_t k) const
    {
        bool is = true;
        #pragma unroll
        for(uint32_t i = 0; i < 8u; i++)
            if(i < k && b[i] == b[k]) is = false;
        return is;
    }
    // the rows with a corner in corner k's bucket
    __device__ __forceinline__ uint32_t rows(uint32_t k) const
    {
        uint32_t m = 0u;
        #pragma unroll
        for(uint32_t i = 0; i < 8u; i++)
            if(b[i] == b[k]) m |= 1u << (i >> 1);
        return m;
    }
};

// Sorting blocks take 4096 samples at a time, a thread four of them. Rows come in
// runs of 32 neighbouring voxels. On a hashed level neighbouring lanes take
// neighbouring rows: those with the same (y, z) stay neighbours in their bucket,
// and k_rc_bucket_grad's gathers share cache lines. On a dense level they take
// rows 32 apart: there lanes of one run would add to the same few entries.
__device__ __forceinline__ uint32_t sort_sample(bool dense, uint32_t first, uint32_t t, uint32_t k)
{
    return first + (dense ? (t & 127u) * 32u + (t >> 7) + 8u * k : t + 1024u * k);
}
// First and last + 1 of a sorting block's samples, in whole 4096s.
__device__ __forceinline__ uint32_t sort_span(uint32_t n)
{
    return ((n + 4095u) / 4096u + gridDim.x - 1u) / gridDim.x * 4096u;
}

// blockIdx.y: the level. The blocks of level 0 also write the unit positions,
// with the divisions by the extent that the other kernels then need not make.
__global__ __launch_bounds__(1024) void k_rc_bucket_count(DNrcNet net, const float* samples, uint32_t n, DNrcActs acts)
{
    __shared__ uint32_t hist[RC_MAX_BUCKETS];
    const uint32_t l = blockIdx.y, t = threadIdx.x;
    const uint32_t buckets = level_buckets(net, l);
    if(buckets == 1u && l != 0u) return;
    if(t < RC_MAX_BUCKETS) hist[t] = 0u;
    __syncthreads();
    const uint32_t N = net.res[l], mask = (1u << net.log2T) - 1u, span = sort_span(n);
    const bool dense = (net.denseMask >> l) & 1u;
    for(uint32_t f = blockIdx.x * span; f < blockIdx.x * span + span; f += 4096u)
        for(uint32_t k = 0; k < 4u; k++)
        {
            const uint32_t s = sort_sample(dense, f, t, k);
            if(s >= n) continue;
            const UnitPos u = unit_pos(net, samples + (size_t)s * RC_SAMPLE);
            if(l == 0u) reinterpret_cast<float4*>(acts.unit)[s] = make_float4(u.v[0], u.v[1], u.v[2], 0.0f);
            if(buckets == 1u) continue;
            const SampleBuckets sb(N, dense, mask, u);
            #pragma unroll
            for(uint32_t c = 0; c < 8u; c++)
                if(sb.first(c)) atomicAdd(&hist[sb.b[c]], 1u);
        }
    __syncthreads();
    if(buckets > 1u && t < RC_MAX_BUCKETS)
        acts.blockCount[(l * RC_SORT_BLOCKS + blockIdx.x) * RC_MAX_BUCKETS + t] = hist[t];
}

__global__ __launch_bounds__(1024) void k_rc_bucket_place(DNrcNet net, uint32_t n, DNrcActs acts)
{
    __shared__ uint32_t next[RC_MAX_BUCKETS], firstHalf;
    const uint32_t l = blockIdx.y, t = threadIdx.x;
    const uint32_t buckets = level_buckets(net, l);
    if(buckets == 1u) return;
    // where this block's share of each bucket starts: the buckets in order, in
    // each the blocks in order
    uint32_t total = 0u, before = 0u, incl = 0u;
    if(t < RC_MAX_BUCKETS)
    {
        const uint32_t* cnt = acts.blockCount + l * RC_SORT_BLOCKS * RC_MAX_BUCKETS + t;
        for(uint32_t b = 0; b < gridDim.x; b++)
        {
            const uint32_t v = cnt[b * RC_MAX_BUCKETS];
            if(b < blockIdx.x) before += v;
            total += v;
        }
        if(blockIdx.x == 0u) acts.bucketCount[l * RC_MAX_BUCKETS + t] = total;
        incl = total;
        for(uint32_t off = 1u; off < 64u; off <<= 1)
        {
            const uint32_t v = __shfl_up(incl, off, 64);
            if((t & 63u) >= off) incl += v;
        }
        if(t == 63u) firstHalf = incl;
    }
    __syncthreads();
    if(t < RC_MAX_BUCKETS) next[t] = incl - total + before + (t >= 64u ? firstHalf : 0u);
    __syncthreads();
    const uint32_t N = net.res[l], mask = (1u << net.log2T) - 1u, span = sort_span(n);
    const bool dense = (net.denseMask >> l) & 1u;
    uint32_t* rec = acts.records + (size_t)l * 8u * n;
    for(uint32_t f = blockIdx.x * span; f < blockIdx.x * span + span; f += 4096u)
        for(uint32_t k = 0; k < 4u; k++)
        {
            const uint32_t s = sort_sample(dense, f, t, k);
            if(s >= n) continue;
            const float4 p = reinterpret_cast<const float4*>(acts.unit)[s];
            const SampleBuckets sb(N, dense, mask, UnitPos{{p.x, p.y, p.z}});
            #pragma unroll
            for(uint32_t c = 0; c < 8u; c++)
                if(sb.first(c)) rec[atomicAdd(&next[sb.b[c]], 1u)] = s * 16u + sb.rows(c);
        }
}

// Sums one slice of a bucket in LDS. Blocks take the slices of all buckets in
// turn; a bucket of one slice is added to the table by plain loads and stores,
// one of several by atomics (consecutive entries: 16 to a cache line). Slices of
// hashed levels are longer: their records hold one row each, mostly, those of
// dense levels up to four.
__device__ __forceinline__ uint32_t slice_records(bool dense) { return dense ? 2048u : 5120u; }

__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8, 8)))
void k_rc_bucket_grad(DNrcNet net, uint32_t n, DNrcActs acts)
{
    __shared__ __align__(16) double acc[2u << RC_BUCKET_LOG2];
    __shared__ uint32_t waveSums[16];
    __shared__ uint32_t item[5];                    // level, bucket, first record, records, slices of the bucket
    static_assert(RC_LEVELS == 16 && RC_MAX_BUCKETS == 128, "a wave per level, two buckets per thread");
    const uint32_t t = threadIdx.x, lane = t & 63u, tl = t >> 6;
    // this thread's two buckets: their records, and the slices of them and of all earlier ones
    const uint32_t tn = level_buckets(net, tl), tslice = slice_records((net.denseMask >> tl) & 1u);
    uint32_t cnt[2], slices[2];
    for(uint32_t k = 0; k < 2u; k++)
    {
        const uint32_t b = 2u * lane + k;
        cnt[k] = b >= tn ? 0u : (tn == 1u ? n : acts.bucketCount[tl * RC_MAX_BUCKETS + b]);
        slices[k] = (cnt[k] + tslice - 1u) / tslice;
    }
    uint32_t start = cnt[0] + cnt[1], before = slices[0] + slices[1];
    for(uint32_t off = 1u; off < 64u; off <<= 1)
    {
        const uint32_t a = __shfl_up(start, off, 64), b = __shfl_up(before, off, 64);
        if(lane >= off) { start += a; before += b; }
    }
    if(lane == 63u) waveSums[tl] = before;
    __syncthreads();
    start -= cnt[0] + cnt[1];
    before -= slices[0] + slices[1];
    uint32_t total = 0u;
    for(uint32_t w = 0; w < 16u; w++)
    {
        if(w == tl) before += total;
        total += waveSums[w];
    }
    const uint32_t mask = (1u << net.log2T) - 1u;
    const uint32_t sums = min(2u << RC_BUCKET_LOG2, 2u << net.log2T);
    for(uint32_t it = blockIdx.x; it < total; it += gridDim.x)
    {
        for(uint32_t k = 0; k < 2u; k++)
        {
            const uint32_t at = before + (k ? slices[0] : 0u);
            if(it < at || it >= at + slices[k]) continue;
            const uint32_t o = (it - at) * tslice;
            item[0] = tl; item[1] = 2u * lane + k; item[2] = start + (k ? cnt[0] : 0u) + o;
            item[3] = min(tslice, cnt[k] - o); item[4] = slices[k];
        }
        for(uint32_t i = t; i < sums / 2u; i += 1024u) reinterpret_cast<double2*>(acc)[i] = make_double2(0.0, 0.0);
        __syncthreads();
        const uint32_t l = item[0], bucket = item[1], first = item[2], count = item[3], parts = item[4];
        const uint32_t N = net.res[l], lo = bucket << RC_BUCKET_LOG2;
        const bool dense = (net.denseMask >> l) & 1u, whole = level_buckets(net, l) == 1u;
        const uint32_t* rec = acts.records + (size_t)l * 8u * n + first;
        const float2* denc = reinterpret_cast<const float2*>(acts.denc) + (size_t)l * n;
        // two records at a time, so that a wave waits for records and then for
        // their samples once per two
        const uint32_t whole32 = (count + 31u) / 32u;               // runs of 32 samples in a slice without records
        for(uint32_t r0 = t; r0 < (whole ? whole32 * 32u : count); r0 += 2048u)
        {
            uint32_t s[2], rows[2];
            float2 d[2];
            float4 p[2];
            #pragma unroll
            for(uint32_t k = 0; k < 2u; k++)
            {
                const uint32_t r = r0 + 1024u * k;
                s[k] = n;
                if(whole)
                {
                    if(r < whole32 * 32u) s[k] = first + (r % whole32) * 32u + r / whole32;
                    rows[k] = 15u;
                }
                else if(r < count)
                {
                    const uint32_t w = rec[r];
                    s[k] = w >> 4;
                    rows[k] = w & 15u;
                }
            }
            #pragma unroll
            for(uint32_t k = 0; k < 2u; k++)
            {
                d[k] = make_float2(0.0f, 0.0f);
                if(s[k] >= n) continue;
                d[k] = denc[s[k]];
                p[k] = reinterpret_cast<const float4*>(acts.unit)[s[k]];
            }
            #pragma unroll
            for(uint32_t k = 0; k < 2u; k++)
            {
                if(d[k].x == 0.0f && d[k].y == 0.0f) continue;     // adding +-0 changes no sum
                const LevelCell c = level_cell(N, UnitPos{{p[k].x, p[k].y, p[k].z}});
                for(uint32_t m = rows[k]; m; m &= m - 1u)
                {
                    const uint32_t j = (uint32_t)__builtin_ctz(m);
                    for(uint32_t x = 0; x < 2u; x++)
                    {
                        const uint32_t i = corner_index(N, dense, mask, c, 2u * j + x);
                        if((i >> RC_BUCKET_LOG2) != bucket) continue;
                        const float w = corner_weight(c, 2u * j + x);
                        double* a = acc + 2u * (i - lo);
                        atomicAdd(a, (double)(w * d[k].x));
                        atomicAdd(a + 1, (double)(w * d[k].y));
                    }
                }
            }
        }
        __syncthreads();
        float* g = net.tabGrad + (((size_t)l << net.log2T) + lo) * 2u;
        if(parts == 1u)
            for(uint32_t i = t; i < sums / 2u; i += 1024u)
            {
                const double2 v = reinterpret_cast<const double2*>(acc)[i];
                if(v.x == 0.0 && v.y == 0.0) continue;
                float2 o = reinterpret_cast<float2*>(g)[i];
                o.x += (float)v.x; o.y += (float)v.y;
                reinterpret_cast<float2*>(g)[i] = o;
            }
        else
            for(uint32_t i = t; i < sums; i += 1024u)
            {
                const float v = (float)acc[i];
                if(v != 0.0f) atomicAdd(g + i, v);
            }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// MLP over 16-sample tiles. Weights in fragment order, staged in LDS by 16-byte
// pieces.

__device__ __forceinline__ void stage_weights(uint16_t* lds, const uint16_t* w, uint32_t threads)
{
    for(uint32_t i = threadIdx.x; i < RC_NPARAM / 8u; i += threads)
        reinterpret_cast<uint4*>(lds)[i] = reinterpret_cast<const uint4*>(w)[i];
}

// A row's third 16-feature input block: normal, albedo, zeros.
__device__ __forceinline__ bf16x4 surface_input(const float* row, uint32_t q)
{
    f32x4 x = {0.0f, 0.0f, 0.0f, 0.0f};
    if(q == 0u) x = f32x4{row[3], row[4], row[5], row[6]};
    else if(q == 1u) x = f32x4{row[7], row[8], 0.0f, 0.0f};
    return to_bf16(x);
}

// A lane's features 4 q + 0..3 of a 16-feature block: two levels' words.
__device__ __forceinline__ bf16x4 level_input(uint32_t even, uint32_t odd)
{
    return __builtin_bit_cast(bf16x4, make_uint2(even, odd));
}

__device__ __forceinline__ void load_input(const uint32_t* x0, uint32_t n, uint32_t sm, const float* row, uint32_t q,
                                           bf16x4 xin[3])
{
    for(uint32_t b = 0; b < 2u; b++)
    {
        const uint32_t* p = x0 + (size_t)(8u * b + 2u * q) * n + sm;
        xin[b] = level_input(p[0], p[n]);
    }
    xin[2] = surface_input(row, q);
}

// One tile. The first layer's third input block is a 16x16x16 product on top of
// the 16x16x32 one. Right behind it, that product has added to an unfinished
// accumulator (wrong elements 0 and 1 of the four: the two instructions take
// different numbers of passes, and the compiler puts no wait between them), so
// all four row blocks go through the K = 32 instruction first: three of them lie
// between a block's two products.
__device__ __forceinline__ void mlp_forward(const uint16_t* W, uint32_t lane, const bf16x4 xin[3], bf16x4 h[3][4],
                                            f32x4& y)
{
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    bf16x4 c[4];
    f32x4 acc[4];
    #pragma unroll
    for(uint32_t mb = 0; mb < 4; mb++) c[mb] = a_frag16(W + RC_OFF_W0 + mb * 768u + 512u, lane);
    #pragma unroll
    for(uint32_t mb = 0; mb < 4; mb++)
        acc[mb] = mfma32(a_frag32(W + RC_OFF_W0 + mb * 768u, lane), xin[0], xin[1], zero);
    __builtin_amdgcn_sched_barrier(0);
    #pragma unroll
    for(uint32_t mb = 0; mb < 4; mb++) acc[mb] = mfma16(c[mb], xin[2], acc[mb]);
    __builtin_amdgcn_sched_barrier(0);
    #pragma unroll
    for(uint32_t mb = 0; mb < 4; mb++) h[0][mb] = relu_bf16(acc[mb]);
    #pragma unroll
    for(uint32_t layer = 1; layer < 3; layer++)
        #pragma unroll
        for(uint32_t mb = 0; mb < 4; mb++)
        {
            const uint16_t* w = W + (layer == 1 ? RC_OFF_W1 : RC_OFF_W2) + mb * 1024u;
            const f32x4 d = mfma32(a_frag32(w, lane), h[layer - 1][0], h[layer - 1][1], zero);
            h[layer][mb] = relu_bf16(mfma32(a_frag32(w + 512, lane), h[layer - 1][2], h[layer - 1][3], d));
        }
    y = mfma32(a_frag32(W + RC_OFF_W3, lane), h[2][0], h[2][1], zero);
    y = mfma32(a_frag32(W + RC_OFF_W3 + 512, lane), h[2][2], h[2][3], y);
}

// Predictions: each lane encodes the four levels whose features it feeds to the
// first layer, so there is one launch and no pass over encoded rows, and no
// scratch memory that calls would share. Bound by the table gathers (a row's 128
// corners with some 85 of them; 10^6 rows at 2^19 entries 171 us, 178 with 128).
// Against encoding all rows in a launch of their own (a level per wave, each XCD two
// levels), both with 128 gathers, 5.7 against 7.5 us at 1008 rows, 17.6 against 22.6
// at 65 536 and 181 against 202 at 10^6; one row per 16 lanes with the weights' LDS
// reads in bank conflict took 13.1, 44.9 and 360.
__global__ __launch_bounds__(256) void k_rc_predict(DNrcNet net, const float* samples, uint32_t n, float* pred)
{
    __shared__ __align__(16) uint16_t W[RC_NPARAM];
    __shared__ uint32_t res[RC_LEVELS];
    stage_weights(W, net.w16, 256u);
    if(threadIdx.x < RC_LEVELS) res[threadIdx.x] = net.res[threadIdx.x];
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u, q = lane >> 4;
    const uint32_t tiles = n / 16u, mask = (1u << net.log2T) - 1u;
    for(uint32_t tile = blockIdx.x * 4u + (threadIdx.x >> 6); tile < tiles; tile += gridDim.x * 4u)
    {
        const uint32_t sm = tile * 16u + (lane & 15u);
        const float* row = samples + (size_t)sm * RC_SAMPLE;
        bf16x4 xin[3], h[3][4];
        f32x4 y;
        const UnitPos u = unit_pos(net, row);
        uint32_t e[4];
        #pragma unroll
        for(uint32_t i = 0; i < 4u; i++)
        {
            // the wave's levels at this step: 8 (i / 2) + 2 q + i mod 2, q = 0..3
            const uint32_t l = 8u * (i >> 1) + 2u * q + (i & 1u);
            const uint32_t kinds = (net.denseMask >> (8u * (i >> 1) + (i & 1u))) & 0x55u;
            if(kinds == 0x55u) e[i] = encode_level<1>(net.tab16, l << net.log2T, res[l], true, mask, u);
            else if(kinds == 0u) e[i] = encode_level<2>(net.tab16, l << net.log2T, res[l], false, mask, u);
            else e[i] = encode_level<0>(net.tab16, l << net.log2T, res[l], (net.denseMask >> l) & 1u, mask, u);
        }
        xin[0] = level_input(e[0], e[1]);
        xin[1] = level_input(e[2], e[3]);
        xin[2] = surface_input(row, q);
        // the weights stay in LDS: held in registers over the tiles (96 of them)
        // they would halve the waves that hide the gathers
        asm volatile("" ::: "memory");
        mlp_forward(W, lane, xin, h, y);
        // y: lane < 16 holds outputs 0..3 of the tile's sample `lane` (3 used);
        // a row may carry an exactly computed term (direct light) in 13..15
        if(lane < 16u)
            reinterpret_cast<float4*>(pred)[sm] =
                make_float4(y[0] + row[13], y[1] + row[14], y[2] + row[15], row[12]);
    }
}

// Forward, backward and weight gradients of training: one tile per wave at a time, the
// RC_MLP_WAVES tiles of a block together for the weight gradients dW = dZ^T X, whose K
// is the samples. Layer by layer the block's dZ and X go to LDS as [feature][sample]
// and each wave multiplies its six 16x16 tiles of the 48 (v_mfma_f32_16x16x32_bf16,
// 32 samples a step), so a wave holds 24 accumulators over all its tiles and neither
// activations nor dZ go to memory: 900 bytes a sample, which a launch of its own used
// to read back (2^17 samples: 41 us against 41 and 47, and 139 where that launch ran
// beside the table gradients).
#define RC_MLP_WAVES 8
// One block a CU (210 VGPRs, 80 KiB of LDS): 41 us per 2^17 samples beside the sorting
// kernels, 69 at 512 blocks.
#define RC_MLP_BLOCKS 256u
enum { RC_SPAN = 16 * RC_MLP_WAVES };          // samples of a block's tiles

// Position in a staged matrix of sample s of feature f: rows of RC_SPAN samples, whose
// 16-byte pieces (8 samples) are permuted by the feature, so that 16 lanes which read
// the same piece of 16 rows meet all banks.
__device__ __forceinline__ uint32_t staged_at(uint32_t f, uint32_t s)
{
    return f * RC_SPAN + (((s >> 3) ^ (f & (RC_SPAN / 8u - 1u))) << 3) + (s & 7u);
}

// Writes a C-layout tile of feature block fb: sample `s` of the block's, features
// 16 fb + 4 q + 0..3.
__device__ __forceinline__ void stage_tile(uint16_t* m, uint32_t fb, uint32_t q, uint32_t s, bf16x4 v)
{
    #pragma unroll
    for(uint32_t i = 0; i < 4u; i++) m[staged_at(16u * fb + 4u * q + i, s)] = (uint16_t)v[i];
}

// acc += A B^T over the block's samples: 16 rows of each of two staged matrices.
__device__ __forceinline__ f32x4 samples_product(const uint16_t* a, uint32_t ab, const uint16_t* b, uint32_t bb,
                                                 uint32_t lane, f32x4 acc)
{
    const uint32_t r = lane & 15u, q = lane >> 4;
    #pragma unroll
    for(uint32_t k = 0; k < RC_SPAN; k += 32u)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(a + staged_at(16u * ab + r, k + 8u * q))),
            __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(b + staged_at(16u * bb + r, k + 8u * q))), acc, 0,
            0, 0);
    return acc;
}

// Adds a C-layout tile of a weight gradient: rows 16 rb + 4 q + 0..3, column 16 cb + lane mod 16.
__device__ __forceinline__ void add_wgrad(float* g, uint32_t ld, uint32_t rb, uint32_t cb, uint32_t lane, f32x4 v)
{
    for(uint32_t i = 0; i < 4u; i++)
        atomicAdd(g + (16u * rb + 4u * (lane >> 4) + i) * ld + 16u * cb + (lane & 15u), v[i]);
}

__global__ __launch_bounds__(64 * RC_MLP_WAVES) void k_rc_mlp(DNrcNet net, const float* samples, uint32_t n,
                                                              float invB, DNrcActs acts)
{
    static_assert(RC_MLP_WAVES == 8, "six tiles of the weight gradients per wave");
    __shared__ __align__(16) uint16_t W[RC_NPARAM];
    __shared__ __align__(16) uint16_t WT[RC_NPARAM];
    __shared__ __align__(16) uint16_t Z[RC_W * RC_SPAN];
    __shared__ __align__(16) uint16_t X[RC_W * RC_SPAN];
    stage_weights(W, net.w16, 64u * RC_MLP_WAVES);
    stage_weights(WT, net.wT16, 64u * RC_MLP_WAVES);
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u, q = lane >> 4, w = threadIdx.x >> 6;
    const uint32_t tiles = n / 16u, at = w * 16u + (lane & 15u);
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    // this wave's tiles: rows w / 2, columns 2 (w mod 2) and the next of W1 and W2; of
    // W0's 4 x 3, waves 0..3 two and waves 4..7 one; of W3's four, waves 4..7 one
    f32x4 g1[2] = {zero, zero}, g2[2] = {zero, zero}, g0a = zero, gb = zero;
    for(uint32_t base = blockIdx.x * RC_MLP_WAVES; base < tiles; base += gridDim.x * RC_MLP_WAVES)
    {
        const uint32_t tile = base + w;
        const bool on = tile < tiles;                   // waves past the end take a tile without weight
        const uint32_t sm = (on ? tile : tiles - 1u) * 16u + (lane & 15u);
        const float* row = samples + (size_t)sm * RC_SAMPLE;
        bf16x4 xin[3], h[3][4];
        f32x4 y;
        load_input(acts.x0, n, sm, row, q, xin);
        mlp_forward(W, lane, xin, h, y);
        // dL/dy = (y - t) / B for valid samples
        f32x4 dy = zero;
        if(on && lane < 16u && row[12] != 0.0f)
            for(int i = 0; i < 3; i++) dy[i] = (y[i] - row[9 + i]) * invB;
        const bf16x4 dyb = to_bf16(dy);
        __syncthreads();                                // the tiles before are multiplied
        stage_tile(Z, 0, q, at, dyb);
        for(uint32_t mb = 0; mb < 4; mb++) stage_tile(X, mb, q, at, h[2][mb]);
        // dH3^T = W3^T dY^T (K = 16 outputs), then through the ReLUs
        bf16x4 dz[4];
        for(uint32_t mb = 0; mb < 4; mb++)
            dz[mb] = relu_grad(mfma16(a_frag16(WT + RC_OFF_W3 + mb * 256u, lane), dyb, zero), h[2][mb]);
        __syncthreads();
        if(w >= 4u) gb = samples_product(Z, 0, X, w - 4u, lane, gb);
        #pragma unroll
        for(int layer = 1; layer >= 0; layer--)
        {
            __syncthreads();
            for(uint32_t mb = 0; mb < 4; mb++)
            {
                stage_tile(Z, mb, q, at, dz[mb]);
                stage_tile(X, mb, q, at, h[layer][mb]);
            }
            // dH_layer^T = W_{layer+1}^T dZ_{layer+1}^T
            const uint16_t* WTl = WT + (layer == 1 ? RC_OFF_W2 : RC_OFF_W1);
            bf16x4 nz[4];
            for(uint32_t mb = 0; mb < 4; mb++)
            {
                f32x4 d = mfma32(a_frag32(WTl + mb * 1024u, lane), dz[0], dz[1], zero);
                d = mfma32(a_frag32(WTl + mb * 1024u + 512u, lane), dz[2], dz[3], d);
                nz[mb] = relu_grad(d, h[layer][mb]);
            }
            __syncthreads();
            for(uint32_t k = 0; k < 2u; k++)
            {
                f32x4& g = layer == 1 ? g2[k] : g1[k];
                g = samples_product(Z, w >> 1, X, 2u * (w & 1u) + k, lane, g);
            }
            for(uint32_t mb = 0; mb < 4; mb++) dz[mb] = nz[mb];
        }
        __syncthreads();
        for(uint32_t mb = 0; mb < 4; mb++) stage_tile(Z, mb, q, at, dz[mb]);
        for(uint32_t ks = 0; ks < 3; ks++) stage_tile(X, ks, q, at, xin[ks]);
        // dX0^T = W0^T dZ1^T, encoded features only (rows 0..31)
        for(uint32_t mb = 0; mb < 2; mb++)
        {
            f32x4 d = mfma32(a_frag32(WT + RC_OFF_W0 + mb * 1024u, lane), dz[0], dz[1], zero);
            d = mfma32(a_frag32(WT + RC_OFF_W0 + mb * 1024u + 512u, lane), dz[2], dz[3], d);
            // features 16 mb + 4 q + 0..3: levels 8 mb + 2 q and the next
            float2* g = reinterpret_cast<float2*>(acts.denc) + (size_t)(8u * mb + 2u * q) * n + sm;
            if(on)
            {
                g[0] = make_float2(d[0], d[1]);
                g[n] = make_float2(d[2], d[3]);
            }
        }
        __syncthreads();
        g0a = samples_product(Z, w & 3u, X, w < 4u ? 0u : 2u, lane, g0a);
        if(w < 4u) gb = samples_product(Z, w, X, 1u, lane, gb);
    }
    if(blockIdx.x * RC_MLP_WAVES >= tiles) return;
    add_wgrad(net.wGrad + RC_OFF_W0, 48u, w & 3u, w < 4u ? 0u : 2u, lane, g0a);
    if(w < 4u) add_wgrad(net.wGrad + RC_OFF_W0, 48u, w, 1u, lane, gb);
    else add_wgrad(net.wGrad + RC_OFF_W3, 64u, 0u, w - 4u, lane, gb);
    for(uint32_t k = 0; k < 2u; k++)
    {
        add_wgrad(net.wGrad + RC_OFF_W1, 64u, w >> 1, 2u * (w & 1u) + k, lane, g1[k]);
        add_wgrad(net.wGrad + RC_OFF_W2, 64u, w >> 1, 2u * (w & 1u) + k, lane, g2[k]);
    }
}

// Adam on FP32 master copies; refreshes the bf16 copies and clears the
// gradients. Weights: one thread per parameter; table: one per entry (2).
__device__ __forceinline__ float adam_one(float& w, float g, float& m, float& v, const DNrcAdam& o)
{
    m = o.beta1 * m + (1.0f - o.beta1) * g;
    v = o.beta2 * v + (1.0f - o.beta2) * g * g;
    w = w - o.lr * (m / o.bias1) / (sqrtf(v / o.bias2) + o.eps);
    return w;
}

__device__ __forceinline__ float ema_one(float& e, float w, const DNrcAdam& o)
{
    e = o.emaDecay * e + (1.0f - o.emaDecay) * w;
    return e * o.emaScale;
}

// A dense level's table ends in entries that no corner has: they are never read, and
// their gradients and moments stay zero, so the step leaves them as they are (45% of
// the table at 2^19 entries and resolutions 16..256). `used`: the entries of a level
// that the step covers, in whole blocks of 256.
struct DNrcUsed { uint32_t blocks[RC_LEVELS + 1]; };     // first block of each level, and their number

// 44 bytes a parameter: bound by HBM.
__global__ __launch_bounds__(256) void k_rc_adam(DNrcNet net, DNrcAdam o, DNrcUsed used)
{
    if(blockIdx.x < RC_NPARAM / 256u)
    {
        const uint32_t i = blockIdx.x * 256u + threadIdx.x;
        float w = net.w32[i], m = net.wM[i], v = net.wV[i], e = net.wE[i];
        adam_one(w, net.wGrad[i], m, v, o);
        net.w32[i] = w; net.wM[i] = m; net.wV[i] = v;
        net.wGrad[i] = 0.0f;
        uint32_t f, t;
        rc_fragment_positions(i, f, t);
        net.w16[f] = net.wT16[t] = f2bf(w);
        net.wE16[f] = f2bf(ema_one(e, w, o));
        net.wE[i] = e;
    }
    else
    {
        const uint32_t b = blockIdx.x - RC_NPARAM / 256u;
        uint32_t l = 0;
        for(uint32_t k = 1; k < RC_LEVELS; k++) l += b >= used.blocks[k] ? 1u : 0u;
        const uint32_t in = (b - used.blocks[l]) * 256u + threadIdx.x;
        if(in >> net.log2T) return;                      // tables smaller than a block
        const size_t i = ((size_t)l << net.log2T) + in;
        float2 w = reinterpret_cast<float2*>(net.tab32)[i];
        float2 g = reinterpret_cast<float2*>(net.tabGrad)[i];
        float2 m = reinterpret_cast<float2*>(net.tabM)[i];
        float2 v = reinterpret_cast<float2*>(net.tabV)[i];
        float2 e = reinterpret_cast<float2*>(net.tabE)[i];
        adam_one(w.x, g.x, m.x, v.x, o);
        adam_one(w.y, g.y, m.y, v.y, o);
        reinterpret_cast<float2*>(net.tab32)[i] = w;
        reinterpret_cast<float2*>(net.tabM)[i] = m;
        reinterpret_cast<float2*>(net.tabV)[i] = v;
        reinterpret_cast<float2*>(net.tabGrad)[i] = make_float2(0.0f, 0.0f);
        net.tab16[i] = f2bf2(w.x, w.y);
        const float ex = ema_one(e.x, w.x, o), ey = ema_one(e.y, w.y, o);
        reinterpret_cast<float2*>(net.tabE)[i] = e;
        net.tabE16[i] = f2bf2(ex, ey);
    }
}

// ---------------------------------------------------------------------------
// training samples: one per lane, a stored voxel of the request list drawn by
// a per-sample hash, lit by the lighting pass's own device functions with
// per-sample random numbers (PCG hash, Jarzynski & Olano, "Hash Functions for
// GPU Rendering", JCGT 2020) instead of the frame-uniform ones.

__device__ __forceinline__ uint32_t pcg(uint32_t v)
{
    uint32_t state = v * 747796405u + 2891336453u;
    uint32_t word = ((state >> ((state >> 28u) + 4u)) ^ state) * 277803737u;
    return (word >> 22u) ^ word;
}

struct SampleRandom {
    uint32_t seed;
    __device__ float u(uint32_t stream, uint32_t k) const
    {
        return (float)(pcg(seed ^ pcg(stream * 0x9E3779B9u + k)) >> 8) * (1.0f / 16777216.0f);
    }
    // uniform in the unit ball by rejection from the cube (as rand_unit_sphere)
    __device__ f3 ball(uint32_t stream) const
    {
        f3 p = splat(0.0f);
        for(uint32_t t = 0; t < 16u; t++)
        {
            p = mk(u(stream, 3 * t) * 2.0f - 1.0f, u(stream, 3 * t + 1) * 2.0f - 1.0f, u(stream, 3 * t + 2) * 2.0f - 1.0f);
            if(dot3(p, p) < 1.0f) return p;
        }
        return p * 0.5f;
    }
    __device__ float glossy_pick(uint32_t sample, uint32_t i) const { return u(100u + sample * 16u + i, 0) * 2.0f - 1.0f; }
    __device__ f3 glossy_dir(uint32_t sample, uint32_t i) const { return ball(200u + sample * 16u + i); }
    __device__ f3 diffuse_dir(uint32_t sample, uint32_t i) const { return ball(300u + sample * 16u + i); }
};

// Locates request slot `slot` (r * 32 + lane): false for an empty lane.
__device__ __forceinline__ bool slot_voxel(const DNlightParams& P, uint32_t slot, const DNchunkRec*& rec,
                                           uint32_t& mapIndex, uint32_t& voxNum, int32_t& sel)
{
    const uint32_t req = P.requests[slot >> 5];
    mapIndex = req >> 4;
    voxNum = (slot & 31u) + (req & 15u) * 32u;
    rec = P.scene.chunks + mapIndex;
    if(voxNum >= rec->numVoxels) return false;
    sel = select_in(rec->mask, voxNum);
    return sel >= 0;
}

__device__ __forceinline__ void write_sample(float* out, f3 pos, const DVoxel& me, f3 target, float valid,
                                             f3 exact = f3{0.0f, 0.0f, 0.0f})
{
    float4* o = reinterpret_cast<float4*>(out);
    o[0] = make_float4(pos.x, pos.y, pos.z, me.normal.x);
    o[1] = make_float4(me.normal.y, me.normal.z, me.albedo.x, me.albedo.y);
    o[2] = make_float4(me.albedo.z, target.x, target.y, target.z);
    o[3] = make_float4(valid, exact.x, exact.y, exact.z);
}

// What the cache learns and what is computed exactly. With fixed direct rays
// (numDirectRays > 0) the ambient and direct terms of a voxel's estimate
// (voxelLighting.comp:255,260) are deterministic: they are evaluated exactly
// and the network learns only the path-traced indirect term. With the
// jittered shadow ray the whole estimate is noisy and the network learns all
// of it.
__device__ __forceinline__ bool direct_is_exact(const DNlightParams& P) { return P.numDirectRays != 0u; }

struct VoxelSite {
    const DNchunkRec* rec;
    uint32_t voxNum;
    int32_t sel;
    DVoxel me;
    f3 p;      // ray origin, voxelLighting.comp:231-232
    f3 pos;    // voxel centre in voxel units
};

__device__ __forceinline__ VoxelSite voxel_site(const DNsceneView& s, const DNchunkRec* rec, uint32_t voxNum, int32_t sel)
{
    VoxelSite v;
    v.rec = rec; v.voxNum = voxNum; v.sel = sel;
    v.me = decompress(s.voxels[rec->voxelIndex + voxNum]);
    const int32_t cx = sel % 8, cy = (sel / 8) % 8, cz = sel / 64;
    v.p = (mk((float)cx, (float)cy, (float)cz) * 0.125f + mk((float)rec->pos[0], (float)rec->pos[1], (float)rec->pos[2])) +
          splat(0.0625f);
    v.p = v.p + splat(0.0625f - DN_EPS) * v.me.normal;
    v.pos = mk((float)(rec->pos[0] * 8 + cx), (float)(rec->pos[1] * 8 + cy), (float)(rec->pos[2] * 8 + cz)) + splat(0.5f);
    return v;
}

__device__ __forceinline__ void site_ctx(const DNlightParams& P, const DNsceneView& s, RayCtx& c, LCtx& L,
                                         uint32_t* maskRows)
{
    ctx_init(c);
    c.maskRow = lane_mask_row(maskRows);
    L.P = &P; L.s = &s; L.c = &c; L.dry = true; L.firstSample = false;
    L.sunDir = ld3(P.sunDir);
    L.sunStrength = ld3(s.sunStrength);
    L.direct = nullptr;
}

// Lane G draws sample g = G mod n of batch k = G / n, with that batch's seed
// seed0 + k * seedStride (the batches of several training steps in one launch).
template <bool OPAQUE>
__global__ __launch_bounds__(256) void k_rc_samples(DNlightParams P, uint32_t n, uint32_t total, uint32_t seed0,
                                                   uint32_t seedStride, float* samples)
{
    __shared__ uint32_t maskRows[DN_MASK_LDS_WORDS(256)];
    const uint32_t G = blockIdx.x * 256u + threadIdx.x;
    if(G >= total) return;
    const uint32_t k = G / n, g = G - k * n;
    const uint32_t seed = seed0 + k * seedStride;
    const uint32_t slots = *P.numRequests * 32u;
    const uint32_t base = pcg(seed ^ pcg(g));
    const DNchunkRec* rec = nullptr;
    uint32_t mapIndex = 0, voxNum = 0;
    int32_t sel = -1;
    bool found = false;
    // first try: slot g & 31 of a request drawn per run of 32 samples (the
    // runs keep a wave's samples in two chunks); then random slots. Over the
    // 32 positions of a run every stored voxel is as likely as any other.
    for(uint32_t t = 0; t < 8u && slots && !found; t++)
    {
        const uint32_t slot = t == 0 ? (pcg(seed ^ pcg((g >> 5) ^ 0x5BD1E995u)) % (slots >> 5)) * 32u + (g & 31u)
                                     : pcg(base + t * 0x68E31DA4u) % slots;
        found = slot_voxel(P, slot, rec, mapIndex, voxNum, sel);
    }
    float* out = samples + (size_t)G * RC_SAMPLE;
    if(!found)
    {
        write_sample(out, splat(0.0f), DVoxel{}, splat(0.0f), 0.0f);
        return;
    }
    const DNsceneView& s = P.scene;
    const VoxelSite v = voxel_site(s, rec, voxNum, sel);
    const DNmat& mat = s.mats[v.me.material];
    RayCtx c;
    LCtx L;
    site_ctx(P, s, c, L, maskRows);
    f3 diff = splat(0.0f);
    if(mat.specular < 1.0f)
    {
        const SampleRandom rng{base};
        diffuse_ray<OPAQUE>(L, v.me.normal + DN_EPS, v.p, v.me, 0, diff, rng);
        if(!direct_is_exact(P))
        {
            diff = diff + ld3(P.ambient);
            f3 dir = vnorm(L.sunDir * P.shadowSoftness + rng.ball(400u)) + DN_EPS;
            DVoxel hv = {};
            f3 ca; float cm;
            f3 pp = v.p;
            if(!light_trace<OPAQUE, !OPAQUE>(s, c, dir, vinv(dir), pp, hv, ca, cm)) diff = diff + (L.sunStrength * cm + ca);
        }
    }
    write_sample(out, v.pos, v.me, diff, 1.0f);
}

// Query rows for every slot of the request list (valid 0 for empty lanes).
template <bool OPAQUE>
__global__ __launch_bounds__(256) void k_rc_gather(DNlightParams P, uint32_t slotsCap, float* samples)
{
    __shared__ uint32_t maskRows[DN_MASK_LDS_WORDS(256)];
    const uint32_t g = blockIdx.x * 256u + threadIdx.x;
    if(g >= slotsCap) return;
    float* out = samples + (size_t)g * RC_SAMPLE;
    const DNchunkRec* rec = nullptr;
    uint32_t mapIndex = 0, voxNum = 0;
    int32_t sel = -1;
    if(g >= *P.numRequests * 32u || !slot_voxel(P, g, rec, mapIndex, voxNum, sel))
    {
        write_sample(out, splat(0.0f), DVoxel{}, splat(0.0f), 0.0f);
        return;
    }
    const DNsceneView& s = P.scene;
    const VoxelSite v = voxel_site(s, rec, voxNum, sel);
    f3 exact = splat(0.0f);
    if(direct_is_exact(P) && s.mats[v.me.material].specular < 1.0f)
    {
        // ambient + the fixed direct rays, as the lighting pass adds them
        RayCtx c;
        LCtx L;
        site_ctx(P, s, c, L, maskRows);
        L.direct = (P.directIn && g < P.directSlots) ? P.directIn + g : nullptr;
        exact = ld3(P.ambient);
        shadow_ray<OPAQUE>(L, v.p, 0, exact);
    }
    write_sample(out, v.pos, v.me, splat(0.0f), 1.0f, exact);
}

// Reference estimate of every slot's irradiance: `per` independent samples per
// thread (per-sample random numbers), `chunks` threads per slot, summed in
// FP64 into acc[slot] (rgb, sample count). With fixed direct rays each sample
// is the exact ambient + direct term plus one path-traced indirect term.
template <bool OPAQUE>
__global__ __launch_bounds__(256) void k_rc_reference(DNlightParams P, uint32_t slotsCap, uint32_t chunks, uint32_t per,
                                                      uint32_t seed, double* acc)
{
    __shared__ uint32_t maskRows[DN_MASK_LDS_WORDS(256)];
    const uint32_t g = blockIdx.x * 256u + threadIdx.x;
    const uint32_t slot = g / chunks, chunk = g % chunks;
    if(slot >= slotsCap || slot >= *P.numRequests * 32u) return;
    const DNchunkRec* rec = nullptr;
    uint32_t mapIndex = 0, voxNum = 0;
    int32_t sel = -1;
    if(!slot_voxel(P, slot, rec, mapIndex, voxNum, sel)) return;
    const DNsceneView& s = P.scene;
    const VoxelSite v = voxel_site(s, rec, voxNum, sel);
    if(s.mats[v.me.material].specular >= 1.0f) return;
    RayCtx c;
    LCtx L;
    site_ctx(P, s, c, L, maskRows);
    const bool exactDirect = direct_is_exact(P);
    f3 exact = splat(0.0f);
    if(exactDirect)
    {
        exact = ld3(P.ambient);
        shadow_ray<OPAQUE>(L, v.p, 0, exact);
    }
    double sx = 0.0, sy = 0.0, sz = 0.0;
    for(uint32_t k = 0; k < per; k++)
    {
        const SampleRandom rng{pcg(seed ^ pcg(slot * 0x9E3779B9u ^ pcg(chunk * per + k)))};
        f3 smp = splat(0.0f);
        diffuse_ray<OPAQUE>(L, v.me.normal + DN_EPS, v.p, v.me, 0, smp, rng);
        if(exactDirect)
            smp = smp + exact;
        else
        {
            smp = smp + ld3(P.ambient);
            f3 dir = vnorm(L.sunDir * P.shadowSoftness + rng.ball(400u)) + DN_EPS;
            DVoxel hv = {};
            f3 ca; float cm;
            f3 pp = v.p;
            if(!light_trace<OPAQUE, !OPAQUE>(s, c, dir, vinv(dir), pp, hv, ca, cm)) smp = smp + (L.sunStrength * cm + ca);
        }
        sx += (double)smp.x; sy += (double)smp.y; sz += (double)smp.z;
    }
    double* a = acc + (size_t)slot * 4u;
    atomicAdd(a + 0, sx);
    atomicAdd(a + 1, sy);
    atomicAdd(a + 2, sz);
    atomicAdd(a + 3, (double)per);
}

__global__ __launch_bounds__(256) void k_accumulate_f64(const float* src, double* dst, size_t n)
{
    for(size_t i = (size_t)blockIdx.x * 256u + threadIdx.x; i < n; i += (size_t)gridDim.x * 256u)
        dst[i] += (double)src[i];
}

inline uint32_t blocks_for(size_t threads, uint32_t cap = 0x7FFFFFFFu)
{
    size_t b = (threads + 255u) / 256u;
    if(b < 1) b = 1;
    return (uint32_t)(b > cap ? cap : b);
}

}  // namespace

int dn_rc_predict(const DNrcNet& net, const float* samples, uint32_t n, float* pred, hipStream_t stream)
{
    if(n == 0 || (n & 15u)) return n ? (int)hipErrorInvalidValue : 0;
    // at most three blocks a CU: more of them evict each other's table lines
    // (10^6 rows, 2^19 entries: 181 us; 188 at 1024 blocks, 190 at 1536), fewer
    // leave small tables waiting (2^14 entries: 120 us; 132 at 512 blocks)
    hipLaunchKernelGGL(k_rc_predict, dim3(blocks_for((size_t)n * 4u, 768)), dim3(256), 0, stream, net, samples, n,
                       pred);
    return (int)hipGetLastError();
}

// Below some 10^4 rows the three sorted launches cost more than the atomics of
// the one (8192 rows, 2^14 / 2^19 entries: 81 / 77 us a step against 73 / 73;
// 16384: 102 / 95 against 114 / 113; 131072: 212 / 217 against 603 / 588). Tables
// above 2^19 entries would need more buckets than a level's scan holds.
bool rc_bucketed(const DNrcNet& net, uint32_t n)
{
    return (1u << net.log2T) <= (uint32_t)RC_MAX_BUCKETS << RC_BUCKET_LOG2 && n >= 12288u && n <= RC_BUCKETED_MAX;
}

int dn_rc_train(const DNrcNet& net, const float* samples, uint32_t n, const DNrcActs& a, hipStream_t stream,
                const DNrcSide* side)
{
    if(n == 0 || (n & 15u)) return n ? (int)hipErrorInvalidValue : 0;
    const uint32_t tiles = n / 16u;
    const bool bucketed = rc_bucketed(net, n);
    // The corner rows are sorted (bound by LDS atomics) beside the encoding (bound by
    // its gathers) and the MLP: they share nothing but the samples. (Sorting the next
    // step's rows beside this step's table gradients and Adam: 2371 against 2275 us per
    // 8 steps of 2^17 rows; the gradients then wait for LDS.)
    hipStream_t ss = stream;
    if(bucketed && side)
    {
        if(hipEventRecord(side->fork, stream) != hipSuccess ||
           hipStreamWaitEvent(side->stream, side->fork, 0) != hipSuccess)
            return (int)hipErrorLaunchFailure;
        ss = side->stream;
    }
    if(bucketed)
    {
        const uint32_t chunks = (n + 4095u) / 4096u;
        const dim3 grid(chunks < RC_SORT_BLOCKS ? chunks : (uint32_t)RC_SORT_BLOCKS, RC_LEVELS);
        hipLaunchKernelGGL(k_rc_bucket_count, grid, dim3(1024), 0, ss, net, samples, n, a);
        hipLaunchKernelGGL(k_rc_bucket_place, grid, dim3(1024), 0, ss, net, n, a);
    }
    hipLaunchKernelGGL(k_rc_encode, dim3(8u * blocks_for(n)), dim3(256), 0, stream, net, samples, n, a.x0);
    const uint32_t spans = (tiles + RC_MLP_WAVES - 1u) / RC_MLP_WAVES;
    hipLaunchKernelGGL(k_rc_mlp, dim3(spans < RC_MLP_BLOCKS ? spans : RC_MLP_BLOCKS), dim3(64u * RC_MLP_WAVES), 0,
                       stream, net, samples, n, 1.0f / (float)n, a);
    if(bucketed && side && (hipEventRecord(side->join, side->stream) != hipSuccess ||
                            hipStreamWaitEvent(stream, side->join, 0) != hipSuccess))
        return (int)hipErrorLaunchFailure;
    if(bucketed)
    {
        // blocks take several slices where there are more than two per CU (all can be
        // resident at once, and each counts the slices only once: 80 us per 2^17 samples
        // against 101 with a block per slice)
        uint32_t blocks = 0;
        for(uint32_t l = 0; l < RC_LEVELS; l++)
        {
            const bool dense = (net.denseMask >> l) & 1u;
            const uint32_t S = net.res[l] + 2u, entries = dense ? S * S * S : 1u << net.log2T;
            const uint32_t buckets = (entries + (1u << RC_BUCKET_LOG2) - 1u) >> RC_BUCKET_LOG2;
            const uint32_t records = dense || buckets == 1u ? n : 4u * n, slice = dense ? 2048u : 5120u;
            blocks += buckets * ((records / buckets + slice - 1u) / slice);
        }
        hipLaunchKernelGGL(k_rc_bucket_grad, dim3(blocks < 512u ? blocks : 512u), dim3(1024), 0, stream, net, n, a);
    }
    else
        // one wave per 16 samples and level
        hipLaunchKernelGGL(k_rc_table_grad, dim3(blocks_for((size_t)RC_LEVELS * ((n + 15u) / 16u) * 64u)), dim3(256), 0,
                       stream, net, samples, n, (const float*)a.denc);
    return (int)hipGetLastError();
}

int dn_rc_adam(const DNrcNet& net, const DNrcAdam& opt, hipStream_t stream)
{
    // with moments of zero a step adds +-0 to a parameter, unless it divides by zero
    const bool skip = opt.bias1 > 0.0f && opt.bias2 > 0.0f && opt.eps > 0.0f && opt.lr >= 0.0f &&
                      opt.lr < INFINITY;
    DNrcUsed used;
    used.blocks[0] = 0;
    for(uint32_t l = 0; l < RC_LEVELS; l++)
    {
        const uint64_t S = net.res[l] + 2ull, T = 1ull << net.log2T;
        const uint64_t entries = skip && ((net.denseMask >> l) & 1u) ? S * S * S : T;
        used.blocks[l + 1] = used.blocks[l] + (uint32_t)((entries + 255u) / 256u);
    }
    hipLaunchKernelGGL(k_rc_adam, dim3(RC_NPARAM / 256u + used.blocks[RC_LEVELS]), dim3(256), 0, stream, net, opt, used);
    return (int)hipGetLastError();
}

int dn_rc_samples(const DNlightParams& p, uint32_t maxRequests, uint32_t n, uint32_t batches, uint32_t seed,
                  uint32_t seedStride, float* samples, hipStream_t stream)
{
    (void)maxRequests;
    if(n == 0 || batches == 0) return 0;
    if((uint64_t)n * batches > 0xFFFFFFFFull) return (int)hipErrorInvalidValue;
    const uint32_t total = n * batches;
    hipLaunchKernelGGL(p.scene.opaque ? k_rc_samples<true> : k_rc_samples<false>, dim3(blocks_for(total)), dim3(256), 0, stream, p, n, total, seed, seedStride,
                       samples);
    return (int)hipGetLastError();
}

int dn_rc_gather(const DNlightParams& p, uint32_t slots, float* samples, hipStream_t stream)
{
    if(slots == 0) return 0;
    hipLaunchKernelGGL(p.scene.opaque ? k_rc_gather<true> : k_rc_gather<false>, dim3(blocks_for(slots)), dim3(256), 0, stream, p, slots, samples);
    return (int)hipGetLastError();
}

int dn_rc_reference(const DNlightParams& p, uint32_t slots, uint32_t samplesPerVoxel, uint32_t seed, double* acc,
                    hipStream_t stream)
{
    if(slots == 0 || samplesPerVoxel == 0) return 0;
    const uint32_t chunks = samplesPerVoxel >= 256u ? 16u : 1u;
    const uint32_t per = (samplesPerVoxel + chunks - 1u) / chunks;
    hipLaunchKernelGGL(p.scene.opaque ? k_rc_reference<true> : k_rc_reference<false>, dim3(blocks_for((size_t)slots * chunks)), dim3(256), 0, stream, p, slots, chunks,
                       per, seed, acc);
    return (int)hipGetLastError();
}

int dn_accumulate_f64(const float* src, double* dst, size_t n, hipStream_t stream)
{
    if(n == 0) return 0;
    hipLaunchKernelGGL(k_accumulate_f64, dim3(blocks_for(n, 4096)), dim3(256), 0, stream, src, dst, n);
    return (int)hipGetLastError();
}
