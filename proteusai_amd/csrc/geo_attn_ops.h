// Operand types of the attention kernels' matrix products: bf16 (default) or fp16 (the reference casts Q, K, V to
// fp16, old/old_scripts/attn/geometric_attn.py:567-569).  Both are 16-bit patterns in memory and in LDS; only the
// matrix instruction, the conversions to the type and the row sum of packed pairs differ.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace proteus_ops {

typedef __bf16   bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16   bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8  __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2  __attribute__((ext_vector_type(2)));
typedef float    floatx16 __attribute__((ext_vector_type(16)));
typedef float    floatx2  __attribute__((ext_vector_type(2)));

template <bool F16> struct Operand;

template <> struct Operand<false> {
    typedef bf16x8 vec8;
    // largest exponential (log2 units) a lazily re-based softmax may hold before it re-bases, and the row-sum alarm
    static constexpr float REBASE = 20.0f, REBASE_SUM = 16777216.0f;
    static __device__ __forceinline__ floatx16 mfma(const uint4 a, const vec8 b, const floatx16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ unsigned pack(const float a, const float b) {
        const floatx2 f = {a, b};
        return __builtin_bit_cast(unsigned, __builtin_convertvector(f, bf16x2));
    }
    // c + the two values packed in w (v_dot2 against ones)
    static __device__ __forceinline__ float add_packed(const unsigned w, const float c) {
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w), __builtin_bit_cast(bf16x2, 0x3f803f80u), c, false);
    }
    // eight raw elements times a power of two (exact)
    static __device__ __forceinline__ vec8 scaled(const uint4 raw, const float s) {
        bf16x8 v = __builtin_bit_cast(bf16x8, raw);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (__bf16)((float)v[e] * s);
        return v;
    }
    static __device__ __forceinline__ vec8 raw8(const uint4 raw) { return __builtin_bit_cast(bf16x8, raw); }
};

template <> struct Operand<true> {
    typedef f16x8 vec8;
    // fp16 ends at 65504: exponentials stay below 2^14
    static constexpr float REBASE = 10.0f, REBASE_SUM = 16384.0f;
    static __device__ __forceinline__ floatx16 mfma(const uint4 a, const vec8 b, const floatx16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ unsigned pack(const float a, const float b) {
        const floatx2 f = {a, b};
        return __builtin_bit_cast(unsigned, __builtin_convertvector(f, f16x2));      // round to nearest even
    }
    static __device__ __forceinline__ float add_packed(const unsigned w, const float c) {
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, w), __builtin_bit_cast(f16x2, 0x3c003c00u), c, false);
    }
    static __device__ __forceinline__ vec8 scaled(const uint4 raw, const float s) {
        f16x8 v = __builtin_bit_cast(f16x8, raw);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (_Float16)((float)v[e] * s);
        return v;
    }
    static __device__ __forceinline__ vec8 raw8(const uint4 raw) { return __builtin_bit_cast(f16x8, raw); }
};

// S = (q . k)/sqrt(d) with q pre-multiplied by the power of two QS (exact in either type) and the remaining factor
// RHO = 1/(sqrt(d) QS) (1 or 2^-1/2) applied to the fp32 product.
template <int D> struct HeadDim;
template <> struct HeadDim<32>  { static constexpr float QS = 0.25f,  RHO = 0.70710678118654752f, INV_SQRT = 0.17677669529663688f; };
template <> struct HeadDim<64>  { static constexpr float QS = 0.125f, RHO = 1.0f,                 INV_SQRT = 0.125f; };
template <> struct HeadDim<128> { static constexpr float QS = 0.125f, RHO = 0.70710678118654752f, INV_SQRT = 0.08838834764831845f; };

// XOR swizzle of the 16-byte chunks of a row-major LDS tile of 16-bit elements with rows of 2 D bytes (chunk c of
// row r sits at slot c ^ tile_swizzle<D>(r)), under which both kinds of reads are free of bank conflicts (64 banks of
// 4 bytes):
//  * 16-byte fragment reads: 16 lanes read one chunk of 16 consecutive rows;
//  * transposing reads (ds_read_b64_tr_b16): 16 lanes read 32 bytes (an even chunk and the next) of four consecutive
//    rows, aligned to four.
// d = 32 (64-byte rows: rows r, r+4, r+8, r+12 share banks): (r >> 2) & 3.
// d = 64 (128-byte rows: the even and the odd rows each share banks): the 8 even and the 8 odd rows of 16 consecutive
//   ones get 8 different values, and rows r, r + 2 of an aligned group of four differ in bits 1..2.
// d = 128 (256-byte rows: all rows share banks): a permutation of r & 15 whose upper three bits differ among four
//   consecutive rows.
template <int D> __device__ __forceinline__ int tile_swizzle(int r);
template <> __device__ __forceinline__ int tile_swizzle<32>(int r)  { return (r >> 2) & 3; }
template <> __device__ __forceinline__ int tile_swizzle<64>(int r)  { return (((r >> 1) & 1) << 2) | ((r >> 2) & 3); }
template <> __device__ __forceinline__ int tile_swizzle<128>(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

// ---- padded batches handed out longest sequence first ----
constexpr int ATTN_LPT_MAX_Z = 64;

// lens[z], zero before: 1 + index of the last unpadded token of sequence z of Z.  Called by all threads of a workgroup.  From 16 tokens on the mask is read 16 bytes at a time
// wherever it lies (a piece is then in at most two sequences), and byte by byte in front of the first multiple of 16 and behind the last: what a launch makes of the lengths
// does not depend on the mask's address.
template <int THREADS>
__device__ __forceinline__ void sequence_lengths(const uint8_t* __restrict__ mask, const int Z, const int N, int* lens)
{
    const int total = Z * N, lead = min((int)(-(uintptr_t)mask & 15), total), pieces = N >= 16 ? (total - lead) >> 4 : 0;
#pragma unroll 4
    for (int p = (int)threadIdx.x; p < pieces; p += THREADS) {
        const int at = lead + 16 * p;
        const uint4 m16 = *reinterpret_cast<const uint4*>(mask + at);
        const unsigned w[4] = {m16.x, m16.y, m16.z, m16.w};
        unsigned usable = 0;                                  // bit e: byte e is zero
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const unsigned zero = ~(((w[e] & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w[e]) & 0x80808080u;       // (bit 7 of a byte that is zero)
            usable |= (((zero >> 7) & 1u) | ((zero >> 14) & 2u) | ((zero >> 21) & 4u) | (zero >> 28)) << (4 * e);
        }
        const int z = at / N, here = (z + 1) * N - at;                               // bytes of the piece in sequence z, the others in z + 1
        const unsigned low = here >= 16 ? usable : usable & ((1u << here) - 1u), high = usable ^ low;
        if (low)  atomicMax(&lens[z], at - z * N + 32 - __builtin_clz(low));
        if (high) atomicMax(&lens[z + 1], 32 - __builtin_clz(high) - here);
    }
    for (int i = (int)threadIdx.x; i < total - 16 * pieces; i += THREADS) {
        const int j = i < lead ? i : i + 16 * pieces;
        if (!mask[j]) atomicMax(&lens[j / N], j % N + 1);
    }
}

// Is token `at` of some sequence padded?  (At most 64 sequences; the same for every wave.)
__device__ __forceinline__ bool some_padded_at(const uint8_t* __restrict__ mask, const int Z, const int N, const int at)
{
    const int lane = threadIdx.x & 63;
    return __builtin_amdgcn_ballot_w64(lane < Z && mask[(size_t)min(lane, Z - 1) * N + at] != 0) != 0;
}

// Workgroup `block_id` of n_tiles * Z * H takes the block_id-th item of the list "live tiles (of OWN tokens) of the longest sequence, tile-major, the heads of a tile
// side by side, those of the next one, ..., then the dead tiles"; tile and zh = (sequence, head) of it.  lens: LDS, left with 1 + index of the last unpadded
// token of every sequence (KNOWN: they are there).  Called by all threads of a workgroup.
template <int THREADS, bool KNOWN = false>
__device__ __forceinline__ void by_length(const uint8_t* __restrict__ key_pad, const int Z, const int N, const int H, const int n_tiles, const int own, const int block_id,
                                          int* lens, int& tile, int& zh)
{
    const int tid = threadIdx.x, lane = tid & 63;
    if (!KNOWN) {
        if (tid < Z) lens[tid] = 0;
        __syncthreads();
        sequence_lengths<THREADS>(key_pad, Z, N, lens);
        __syncthreads();
    }
    const int mine = lane < Z ? lens[lane] : 0;
    int rank = lane < Z ? 0 : lane;
    for (int u = 0; u < Z; ++u) {
        const int o = __builtin_amdgcn_readlane(mine, u);
        if (lane < Z) rank += (o > mine || (o == mine && u < lane)) ? 1 : 0;
    }
    // lane r: the sequence of rank r, its live tiles, and the workgroups of all up to it
    const int item = __builtin_amdgcn_ds_permute(rank << 2, lane);
    const int tiles = (__builtin_amdgcn_ds_permute(rank << 2, mine) + own - 1) / own;
    auto up_to = [&](int n) {
        for (int o = 1; o < 64; o *= 2) { const int below = __shfl_up(n, o); if (lane >= o) n += below; }
        return n;
    };
    // (the list laid over the launch as a snake, every second row of 256 workgroups reversed: workgroups b and
    // b + 256 share a compute unit while the launch fills the chip, and get a long and a short item)
    int rem = block_id;
    {
        const int total = n_tiles * Z * H, row0 = block_id - block_id % 256;
        const int rowlen = min(total - row0, 256);
        if ((block_id / 256) & 1) rem = row0 + (rowlen - 1 - (block_id - row0));
    }
    int cnt = lane < Z ? tiles * H : 0, sum = up_to(cnt), first = 0;
    const int live = __builtin_amdgcn_readlane(sum, 63);
    const bool dead = rem >= live;
    if (dead) {
        rem -= live;
        cnt = lane < Z ? (n_tiles - tiles) * H : 0;
        sum = up_to(cnt);
    }
    const int sel = __builtin_ctzll(__builtin_amdgcn_ballot_w64(rem < sum));        // (the list has a place for every workgroup)
    if (dead) first = __builtin_amdgcn_readlane(tiles, sel);
    rem -= __builtin_amdgcn_readlane(sum, sel) - __builtin_amdgcn_readlane(cnt, sel);
    const int zsel = __builtin_amdgcn_readlane(item, sel);
    rem = __builtin_amdgcn_readfirstlane(rem);
    tile = __builtin_amdgcn_readfirstlane(first) + rem / H;
    zh = zsel * H + rem % H;
}

}  // namespace proteus_ops
