// kquant.hip -- GGUF K-quant weights: Q4_K and Q6_K against Q8_K
// activations (the reference's integer-activation dots), Q5_K against fp32
// activations (its dequant-in-dot form), the activation quantizer, and the
// row gather of the embedding. Bit-exact to the reference.
//
//   quantize_row_q8_K      nm/src/quant_i8.hpp:31-64
//   vec_dot_q4_K_q8_K      nm/src/quant_i8.hpp:146-191 (scalar form)
//   vec_dot_q6_K_q8_K      nm/src/quant_i8.hpp:239-278 (scalar form)
//   dot_block_q5_K         nm/src/quant.hpp:207-229
//   Weight::matvec/matmul  nm/src/quant_i8.hpp:352-383, 415-495
//   dequant_to_f32         nm/src/quant.hpp:322-395
//
// Weights are repacked once at load (kq_pack_kernel): within a super-block the
// bytes of the four positions 32j + 8i + l (i = 0..3) that share sub-block j
// and residue l = p % 8 -- the positions whose products the reference adds
// into one of its eight sums -- become one dword, so each such group is one
// 4-way int8 dot; the blocks are laid out so that each wave's weight loads
// are contiguous (the tiled layout below). A Q8_K
// activation row is K/256 GGUF blocks of 292 bytes {fp32 d, int8 qs[256],
// int16 bsums[16]} followed by the same residue regrouping of its int8.
//
// Exactness: per super-block the reference forms eight int32 sums aux[l]
// (each product weighted by its sub-block's integer scale) and, for Q4_K, the
// integer mins term; all of that is exact, so any order gives the same
// integers. The fp32 part runs per output in block order exactly as written:
// d = fp16(w.d) * x.d; sums[l] += d * float(aux[l]); (Q4_K)
// sumf -= (fp16(w.dmin) * x.d) * float(summin); then sumf += sums[0..7].
#include <algorithm>

#include "hero/device.hpp"
#include "hero/errors.hpp"
#include "hero/kernels.hpp"

namespace hero {

namespace {

constexpr int kQ8KBytes = 292;
constexpr int kKqThreads = 256;

// ---- the packed weight layout -------------------------------------------------------
// A workgroup owns R = 256 / nb consecutive output rows (a tile) and its lane
// `item` = b * R + r the super-block b of row r. Packed, each tile's blocks are
// stored wave by wave (64 items) as structure-of-arrays: 16-byte chunk u of the
// 64 blocks of a wave is 1 KiB of contiguous memory, so each weight load of a
// wave is one coalesced access. Chunks per block: Q4_K 9 (16-byte header, 8 of
// residue-regrouped quants), Q5_K 11 (the GGUF bytes), Q6_K 13 (8 of ql, 4 of
// qh, both regrouped, 1 of scales) plus a plane of fp16 d, one per slot.
__host__ __device__ inline int kq_rows_per_tile(int64_t K) { return int(K / 256) >= kKqThreads ? 1 : kKqThreads / int(K / 256); }
__host__ __device__ inline int kq_waves_per_tile(int64_t K) { return (kq_rows_per_tile(K) * int(K / 256) + 63) / 64; }
__host__ __device__ inline int kq_chunks(int type) { return type == 12 ? 9 : type == 13 ? 11 : 13; }
// slot of block (n, b): (tile * waves_per_tile + wave) * 64 + lane
__host__ __device__ inline int64_t kq_slot(int64_t n, int b, int64_t K) {
    const int R = kq_rows_per_tile(K);
    const int64_t t = n / R;
    const int item = b * R + int(n % R);
    return (t * kq_waves_per_tile(K) + item / 64) * 64 + item % 64;
}
// uint4 index of chunk u of the block in `slot`
__host__ __device__ inline int64_t kq_chunk_index(int64_t slot, int u, int U) { return ((slot / 64) * U + u) * 64 + slot % 64; }
__host__ __device__ inline int64_t kq_slots(int64_t N, int64_t K) {
    const int R = kq_rows_per_tile(K);
    return (N + R - 1) / R * kq_waves_per_tile(K) * 64;
}

__device__ __forceinline__ int nearest_int_magic(float v) {
    const float t = v + 12582912.f;  // 1.5 * 2^23: rounds to nearest, ties to even
    return (__float_as_int(t) & 0x007fffff) - 0x00400000;
}

// One wave per 256-element block; lane i holds elements 4i .. 4i+3.
// Besides the GGUF block, each block's 256 int8 are written regrouped (xt):
// per 32-element sub-block j, dword 8j + l = bytes (q[32j+l], q[32j+8+l],
// q[32j+16+l], q[32j+24+l]) -- the four positions that share a Q4_K integer
// sum and scale, so a Q4_K block's terms are 4-way int8 dots.
__global__ __launch_bounds__(64) void quantize_q8_K_kernel(const float* __restrict__ x, uint8_t* __restrict__ act, uint32_t* __restrict__ xt,
                                                           int64_t nblocks) {
    __shared__ uint32_t qsh[64];
    const int64_t blk = blockIdx.x;
    if (blk >= nblocks) return;
    const int lane = threadIdx.x;
    const float4 v = reinterpret_cast<const float4*>(x + blk * 256)[lane];
    const float e[4] = {v.x, v.y, v.z, v.w};
    // first element of largest magnitude (strict >, in index order)
    float amax = 0.f;
    int idx = 1 << 30;
    for (int u = 0; u < 4; ++u) {
        const float a = fabsf(e[u]);
        if (a > amax) amax = a, idx = 4 * lane + u;
    }
    for (int off = 32; off > 0; off >>= 1) {
        const float oa = __shfl_xor(amax, off);
        const int oi = __shfl_xor(idx, off);
        if (oa > amax || (oa == amax && oi < idx)) amax = oa, idx = oi;
    }
    uint8_t* out = act + blk * kQ8KBytes;
    if (amax == 0.f) {  // the zero block: d = 0, quants and sums 0
        reinterpret_cast<uint32_t*>(out)[lane] = 0u;
        if (lane < 9) reinterpret_cast<uint32_t*>(out + 256)[lane] = 0u;
        xt[blk * 64 + lane] = 0u;
        return;
    }
    const float mx = __shfl(e[idx & 3], idx >> 2);
    const float iscale = -127.f / mx;
    int q[4];
    for (int u = 0; u < 4; ++u) q[u] = min(127, nearest_int_magic(iscale * e[u]));
    const uint32_t packed = (uint32_t(q[0]) & 0xFF) | ((uint32_t(q[1]) & 0xFF) << 8) | ((uint32_t(q[2]) & 0xFF) << 16) | (uint32_t(q[3]) << 24);
    reinterpret_cast<uint32_t*>(out + 4)[lane] = packed;
    qsh[lane] = packed;
    __syncthreads();
    {
        const uint8_t* qb = reinterpret_cast<const uint8_t*>(qsh) + 32 * (lane >> 3) + (lane & 7);
        xt[blk * 64 + lane] = uint32_t(qb[0]) | (uint32_t(qb[8]) << 8) | (uint32_t(qb[16]) << 16) | (uint32_t(qb[24]) << 24);
    }
    int s = q[0] + q[1] + q[2] + q[3];  // sums of 16 = four lanes
    s += __shfl_xor(s, 1);
    s += __shfl_xor(s, 2);
    if ((lane & 3) == 0) reinterpret_cast<int16_t*>(out + 260)[lane >> 2] = int16_t(s);
    if (lane == 0) reinterpret_cast<float*>(out)[0] = 1.f / iscale;
}

// Sign-extend four packed 6-bit values (bytes 0..63) minus 32 to int8:
// t = q ^ 32 has its sign in bit 5; the top two bits copy it (0x20 * 6 = 0xC0).
__device__ __forceinline__ uint32_t sext6_minus32(uint32_t q) {
    const uint32_t t = q ^ 0x20202020u;
    return t | ((t & 0x20202020u) * 6u);
}

// get_scale_min_k4 (nm/src/quant.hpp:153-162): 6-bit scale and min of sub-block j
__device__ __forceinline__ void scale_min_k4(const uint8_t* q, int j, int& sc, int& m) {
    if (j < 4) {
        sc = q[j] & 63;
        m = q[j + 4] & 63;
    } else {
        sc = (q[j + 4] & 0xF) | ((q[j - 4] >> 6) << 4);
        m = (q[j + 4] >> 4) | ((q[j] >> 6) << 4);
    }
}

// the same from the 12 packed bytes held as three dwords (j compile-time)
__device__ __forceinline__ void scale_min_k4_w(const uint32_t (&h)[3], int j, int& sc, int& m) {
    auto byte = [&](int i) { return int((h[i >> 2] >> (8 * (i & 3))) & 0xFFu); };
    if (j < 4) {
        sc = byte(j) & 63;
        m = byte(j + 4) & 63;
    } else {
        sc = (byte(j + 4) & 0xF) | ((byte(j - 4) >> 6) << 4);
        m = (byte(j + 4) >> 4) | ((byte(j) >> 6) << 4);
    }
}
// int8 scale g of 16 held as four dwords (g compile-time), sign-extended
__device__ __forceinline__ int scale_i8_w(const uint32_t (&w)[4], int g) { return int(w[g >> 2] << (24 - 8 * (g & 3))) >> 24; }

constexpr int kKqTile = 4;  // activation rows per pass of the K-quant GEMM

// Q4_K / Q6_K GEMM over packed weights (kq_pack_kernel) and Q8_K activations.
//
// A workgroup owns R consecutive output rows; lane (b, r) = (tid / R, tid % R)
// holds super-block b of row n0 + r in registers for the whole kernel (each
// weight byte is read once per workgroup) and walks the workgroup's
// activation rows kKqTile at a time: per row it forms the block's eight
// residue sums aux[l] (exact integers, dot4 over the residue-grouped bytes)
// and the reference's per-block fp32 products d * aux[l] (and, for Q4_K,
// dmin * sum_of_mins), leaving them in shared memory; then lane (row, r)
// chains row r's blocks in order: sums[l] += P[b][l]; sumf -= Q[b]; and
// finally sumf += sums[0..7] (nm/src/quant_i8.hpp:146-191, 239-278).
// grid (ceil(N / R), ceil(M / rows_per_group)); R * nb <= 256.
// PER_ROW (the one-row form, M = 1): the weights are decoded in the row loop
// rather than once before it, which keeps the kernel at 104 / 112 VGPRs
// instead of 132 / 189 (Q4_K / Q6_K) and so four workgroups per CU, and each
// output's nine chains run on lanes of their own. Q4_K K = 12288 x 4096 rows:
// 17.5 -> 12.0 us; Q6_K 12288 x 4096: 17.8 -> 14.9 us. With several rows per
// workgroup the decode-once form and one lane per output are faster.
template <int TYPE, bool PER_ROW>
__global__ __launch_bounds__(kKqThreads) void kq_gemm_kernel(const uint8_t* __restrict__ w, const uint8_t* __restrict__ act, const uint32_t* __restrict__ xt,
                                                             float* __restrict__ y, const float* __restrict__ resid, int64_t M, int64_t N, int K, int64_t ldy,
                                                             int R, int rows_per_group) {
    extern __shared__ float terms[];  // [kKqTile][R * nb][T]
    constexpr int T = TYPE == 12 ? 9 : 8;
    const int nb = K >> 8, tid = threadIdx.x, items = R * nb;
    const int64_t n0 = int64_t(blockIdx.x) * R;
    const int64_t m_begin = int64_t(blockIdx.y) * rows_per_group;
    const int64_t m_end = min(M, m_begin + rows_per_group);
    const int b = tid / R, r = tid % R;
    const bool active = tid < items && n0 + r < N;
    // this lane's slot: tile blockIdx.x, item tid
    const int64_t slot = (int64_t(blockIdx.x) * ((items + 63) / 64) + tid / 64) * 64 + tid % 64;

    // the block: Q4_K 16-byte header (d, dmin, packed scales) + 32 residue
    // dwords; Q6_K 32 low-nibble dwords, 16 high-bit dwords, 16 int8 scales, d
    // scales stay packed (Q4_K: 12 bytes, Q6_K: 16 int8) and are unpacked where used
    uint32_t q[TYPE == 12 ? 32 : 48];
    uint32_t hs[3] = {0u, 0u, 0u}, s6[4] = {0u, 0u, 0u, 0u};
    int scv[TYPE == 12 ? 8 : 16], mnv[8];  // !PER_ROW: the scales unpacked once
    float wd = 0.f, wdmin = 0.f;
    if (active) {
        const uint4* w4 = reinterpret_cast<const uint4*>(w);
        if constexpr (TYPE == 12) {
            const uint4* src = w4 + kq_chunk_index(slot, 0, 9);  // chunk u at src[64 u]
            const uint4 hdr = src[0];
            hs[0] = hdr.y, hs[1] = hdr.z, hs[2] = hdr.w;
            if constexpr (!PER_ROW) {
#pragma unroll
                for (int j = 0; j < 8; ++j) scale_min_k4_w(hs, j, scv[j], mnv[j]);
            }
            wd = half_bits_to_f32(uint16_t(hdr.x & 0xFFFF));
            wdmin = half_bits_to_f32(uint16_t(hdr.x >> 16));
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint4 v = src[64 * (1 + i)];
                q[4 * i] = v.x, q[4 * i + 1] = v.y, q[4 * i + 2] = v.z, q[4 * i + 3] = v.w;
            }
        } else {
            const uint4* src = w4 + kq_chunk_index(slot, 0, 13);
#pragma unroll
            for (int i = 0; i < 12; ++i) {
                const uint4 v = src[64 * i];
                q[4 * i] = v.x, q[4 * i + 1] = v.y, q[4 * i + 2] = v.z, q[4 * i + 3] = v.w;
            }
            const uint4 sv = src[64 * 12];
            s6[0] = sv.x, s6[1] = sv.y, s6[2] = sv.z, s6[3] = sv.w;
            if constexpr (!PER_ROW) {
#pragma unroll
                for (int g = 0; g < 16; ++g) scv[g] = scale_i8_w(s6, g);
            }
            const uint16_t* dplane = reinterpret_cast<const uint16_t*>(w4 + kq_slots(N, K) * 13);
            wd = half_bits_to_f32(dplane[slot]);
        }
    }

    for (int64_t mt = m_begin; mt < m_end; mt += kKqTile) {
        const int mrows = int(min<int64_t>(kKqTile, m_end - mt));
        if (active) {
#pragma unroll 1
            for (int mi = 0; mi < mrows; ++mi) {
                const int64_t ab = (mt + mi) * nb + b;
                const float xd = *reinterpret_cast<const float*>(act + ab * kQ8KBytes);
                const uint4* xv = reinterpret_cast<const uint4*>(xt + ab * 64);
                int aux[8] = {0, 0, 0, 0, 0, 0, 0, 0};
                float* t = terms + (int64_t(mi) * items + tid) * T;
                if constexpr (PER_ROW) {
                    // opaque to the compiler: the decode below stays in the row loop
                    if constexpr (TYPE == 12) {
                        asm volatile("" : "+v"(hs[0]), "+v"(hs[1]), "+v"(hs[2]));
                    } else {
                        asm volatile("" : "+v"(s6[0]), "+v"(s6[1]), "+v"(s6[2]), "+v"(s6[3]));
                    }
#pragma unroll
                    for (int i = 0; i < (TYPE == 12 ? 32 : 48); ++i) asm volatile("" : "+v"(q[i]));
                }
                if constexpr (TYPE == 12) {
                    if constexpr (PER_ROW) {
                        // the activation's 64 bytes for step c are read one step ahead of their use
                        uint4 xa[4], xb[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) xa[k] = xv[k];
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            if (c < 3) {
#pragma unroll
                                for (int k = 0; k < 4; ++k) xb[k] = xv[4 * (c + 1) + k];
                            }
                            __builtin_amdgcn_sched_barrier(0);
                            const uint32_t xlo[8] = {xa[0].x, xa[0].y, xa[0].z, xa[0].w, xa[1].x, xa[1].y, xa[1].z, xa[1].w};
                            const uint32_t xhi[8] = {xa[2].x, xa[2].y, xa[2].z, xa[2].w, xa[3].x, xa[3].y, xa[3].z, xa[3].w};
                            int s0, s1, m_unused;
                            scale_min_k4_w(hs, 2 * c, s0, m_unused);
                            scale_min_k4_w(hs, 2 * c + 1, s1, m_unused);
#pragma unroll
                            for (int l = 0; l < 8; ++l) {
                                const uint32_t g = q[8 * c + l];
                                aux[l] += s0 * dot4_i8(int(g & 0x0F0F0F0Fu), int(xlo[l]), 0);
                                aux[l] += s1 * dot4_i8(int((g >> 4) & 0x0F0F0F0Fu), int(xhi[l]), 0);
                            }
                            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                            for (int k = 0; k < 4; ++k) xa[k] = xb[k];
                        }
                    } else {
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            const uint4 xl0 = xv[4 * c], xl1 = xv[4 * c + 1], xh0 = xv[4 * c + 2], xh1 = xv[4 * c + 3];
                            const uint32_t xlo[8] = {xl0.x, xl0.y, xl0.z, xl0.w, xl1.x, xl1.y, xl1.z, xl1.w};
                            const uint32_t xhi[8] = {xh0.x, xh0.y, xh0.z, xh0.w, xh1.x, xh1.y, xh1.z, xh1.w};
#pragma unroll
                            for (int l = 0; l < 8; ++l) {
                                const uint32_t g = q[8 * c + l];
                                aux[l] += scv[2 * c] * dot4_i8(int(g & 0x0F0F0F0Fu), int(xlo[l]), 0);
                                aux[l] += scv[2 * c + 1] * dot4_i8(int((g >> 4) & 0x0F0F0F0Fu), int(xhi[l]), 0);
                            }
                        }
                    }
                    const uint32_t* bw = reinterpret_cast<const uint32_t*>(act + ab * kQ8KBytes + 260);  // 16 int16 sums
                    int sumi = 0;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const uint32_t v = bw[i];
                        int mi;
                        if constexpr (PER_ROW) {
                            int sc_unused;
                            scale_min_k4_w(hs, i, sc_unused, mi);
                        } else {
                            mi = mnv[i];
                        }
                        sumi += int(int16_t(v & 0xFFFF)) * mi;  // sums 2i and 2i+1 share min i
                        sumi += int(int16_t(v >> 16)) * mi;
                    }
                    const float d = wd * xd;
#pragma unroll
                    for (int l = 0; l < 8; ++l) t[l] = d * float(aux[l]);
                    const float dmin = wdmin * xd;
                    t[8] = dmin * float(sumi);
                } else {
                    if constexpr (PER_ROW) {
                        // the activation's 32 bytes for step j are read one step ahead of their use
                        uint4 xa[2] = {xv[0], xv[1]}, xb[2];
#pragma unroll
                        for (int j = 0; j < 8; ++j) {
                            if (j < 7) xb[0] = xv[2 * j + 2], xb[1] = xv[2 * j + 3];
                            __builtin_amdgcn_sched_barrier(0);
                            const int cp = 2 * (j / 4) + (j % 2), nib = 4 * ((j % 4) / 2), hh = j / 4, sh = 2 * (j % 4);
                            const uint32_t xs[8] = {xa[0].x, xa[0].y, xa[0].z, xa[0].w, xa[1].x, xa[1].y, xa[1].z, xa[1].w};
                            const int s0 = scale_i8_w(s6, 2 * j), s1 = scale_i8_w(s6, 2 * j + 1);
#pragma unroll
                            for (int l = 0; l < 8; ++l) {
                                const uint32_t lo = (q[8 * cp + l] >> nib) & 0x0F0F0F0Fu;
                                const uint32_t hi = ((q[32 + 8 * hh + l] >> sh) & 0x03030303u) << 4;
                                const uint32_t a = sext6_minus32(lo | hi);
                                // bytes 0, 1: positions of group 2j; bytes 2, 3: group 2j + 1
                                aux[l] += s0 * dot4_i8(int(a & 0x0000FFFFu), int(xs[l]), 0);
                                aux[l] += s1 * dot4_i8(int(a & 0xFFFF0000u), int(xs[l]), 0);
                            }
                            __builtin_amdgcn_sched_barrier(0);
                            xa[0] = xb[0], xa[1] = xb[1];
                        }
                    } else {
#pragma unroll
                        for (int j = 0; j < 8; ++j) {
                            const int cp = 2 * (j / 4) + (j % 2), nib = 4 * ((j % 4) / 2), hh = j / 4, sh = 2 * (j % 4);
                            const uint4 x0 = xv[2 * j], x1 = xv[2 * j + 1];
                            const uint32_t xs[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
                            for (int l = 0; l < 8; ++l) {
                                const uint32_t lo = (q[8 * cp + l] >> nib) & 0x0F0F0F0Fu;
                                const uint32_t hi = ((q[32 + 8 * hh + l] >> sh) & 0x03030303u) << 4;
                                const uint32_t a = sext6_minus32(lo | hi);
                                // bytes 0, 1: positions of group 2j; bytes 2, 3: group 2j + 1
                                aux[l] += scv[2 * j] * dot4_i8(int(a & 0x0000FFFFu), int(xs[l]), 0);
                                aux[l] += scv[2 * j + 1] * dot4_i8(int(a & 0xFFFF0000u), int(xs[l]), 0);
                            }
                        }
                    }
                    const float d = wd * xd;
#pragma unroll
                    for (int l = 0; l < 8; ++l) t[l] = d * float(aux[l]);
                }
            }
        }
        __syncthreads();
        if constexpr (PER_ROW) {
            // 16 lanes per output: lane l < 8 of the group runs sums[l] over the
            // blocks, lane 8 (Q4_K) the mins chain 0 - Q[0] - Q[1] ..., and the
            // group's first lane then forms sumf += sums[0..7] in order: the
            // same operations one lane per output does below
            constexpr int NC = TYPE == 12 ? 9 : 8;  // chains per output
            const int lane = tid & 63;
            for (int idx0 = 0; idx0 < mrows * R * 16; idx0 += kKqThreads) {
                const int idx = idx0 + tid, oi = idx >> 4, part = idx & 15;
                const int mi = oi / R, rr = oi % R;
                const bool out_live = oi < mrows * R && n0 + rr < N;
                float v = 0.f;
                if (out_live && part < NC) {
                    const float* t = terms + (int64_t(mi) * items + rr) * T + part;
                    const bool mins = part == 8;
                    const int step = R * T;
#pragma unroll 4
                    for (int bb = 0; bb < nb; ++bb) {
                        const float x = t[bb * step];
                        v = mins ? v - x : v + x;
                    }
                }
                float c[NC];
#pragma unroll
                for (int l = 0; l < NC; ++l) c[l] = __shfl(v, (lane & ~15) + l);
                if (out_live && part == 0) {
                    float sumf = TYPE == 12 ? c[NC - 1] : 0.f;
#pragma unroll
                    for (int l = 0; l < 8; ++l) sumf += c[l];
                    const int64_t o = (mt + mi) * ldy + n0 + rr;
                    y[o] = resid ? resid[o] + sumf : sumf;
                }
            }
        } else {
            for (int idx = tid; idx < mrows * R; idx += kKqThreads) {
                const int mi = idx / R, rr = idx % R;
                const int64_t n = n0 + rr;
                if (n >= N) continue;
                float sums[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                float sumf = 0.f;
                for (int bb = 0; bb < nb; ++bb) {
                    const float* t = terms + (int64_t(mi) * items + bb * R + rr) * T;
#pragma unroll
                    for (int l = 0; l < 8; ++l) sums[l] += t[l];
                    if constexpr (TYPE == 12) sumf -= t[8];
                }
#pragma unroll
                for (int l = 0; l < 8; ++l) sumf += sums[l];
                const int64_t o = (mt + mi) * ldy + n;
                y[o] = resid ? resid[o] + sumf : sumf;
            }
        }
        __syncthreads();
    }
}

// ---- Q4_K / Q6_K products of several activation rows, on the matrix cores ----------------
// Per (output, super-block) the reference forms eight integer sums, one per
// residue l = position mod 8, and chains each in fp32. A residue's sum is a
// 32-term product: sum over (sub-block j, i) of (scale_j * q) * x. The scaled
// weights are integers of at most 13 bits and x of 8, so fp16 operands hold
// them exactly and every partial sum stays below 2^24: the fp32 accumulator of
// an fp16 MFMA is the integer itself, already converted (32 * 4096 * 127 <
// 2^24). Q4_K's scale * q <= 945 is one fp16; Q6_K's needs two, q = lo4 + 16
// (hi2 - 2): lo4 * scale / 16 and (hi2 - 2) * scale, against x * 16.
//
// A workgroup owns 32 MT activation rows x 32 NT weight rows and wave l its
// residue l: it decodes exactly the weights and activations of that residue
// (nothing is decoded twice in a workgroup), multiplies them and runs the
// outputs' sums[l] chains in its registers: acc += d * aux, super-blocks in
// order. d = w.d * x.d comes as a 32 x 32 x 1 fp32 MFMA, one correctly rounded
// product per output. Q4_K's mins term is a ninth sum over the sixteen sums of
// 16 (|sum| <= 2032, exact in fp16), one tile on each of the first MT * NT
// waves. At the end the waves' chains meet in shared memory and one lane per
// output adds them in the reference's order. The raw blocks of the next
// super-block are staged through shared memory (plane-major, so each wave
// reads its residue's words) while the current one is multiplied.
//
// Bound: vector instructions. Per wave and super-block of a 64 x 64 tile 128
// multiplies and adds run the chains; decoding, staging and addresses take ~230
// more of the half-rate kinds (packed fp16, perm, and-or), the MFMAs (16 or 8
// per wave, plus two fp32 ones that share the vector units) mostly run beside
// them. Measured with the quantizer: Q6_K 512 rows x 4096, K 12288 2426 -> 198
// us, Q4_K 509 rows x 4096, K 4096 410 -> 63 us (before: 4-way integer dots,
// one lane per super-block and row, one chain lane per output).
using h2_t = _Float16 __attribute__((ext_vector_type(2)));
using h8_t = _Float16 __attribute__((ext_vector_type(8)));
using f16v_t = float __attribute__((ext_vector_type(16)));
using f32v_t = float __attribute__((ext_vector_type(32)));

__device__ __forceinline__ h2_t as_h2(uint32_t v) { return __builtin_bit_cast(h2_t, v); }
__device__ __forceinline__ uint32_t as_u32(h2_t v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ h2_t h2_fma(h2_t a, h2_t b, h2_t c) { return __builtin_elementwise_fma(a, b, c); }
__device__ __forceinline__ h2_t h2_of(float v) { return h2_t{_Float16(v), _Float16(v)}; }
__device__ __forceinline__ h8_t h8_of(h2_t a, h2_t b, h2_t c, h2_t d) {
    const uint4 v = make_uint4(as_u32(a), as_u32(b), as_u32(c), as_u32(d));
    return __builtin_bit_cast(h8_t, v);
}
// 1024 + byte, as fp16, of bytes 0 and 2 (even) or 1 and 3 (odd) of a dword
__device__ __forceinline__ h2_t bytes_even(uint32_t v) { return as_h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04020400u)); }
__device__ __forceinline__ h2_t bytes_odd(uint32_t v) { return as_h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04030401u)); }
// 1024 + byte e of a dword, in both halves
__device__ __forceinline__ h2_t byte_twice(uint32_t v, int e) { return as_h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04000400u | uint32_t(e) * 0x00010001u)); }

constexpr int kMmThreads = 512;  // eight waves, one per residue
__device__ __forceinline__ uint32_t mm_chunk_index(uint32_t slot, int u, int U) { return ((slot / 64) * U + u) * 64 + slot % 64; }

template <int TYPE, int MT, int NT>
struct KqMmShared {
    static constexpr int BM = 32 * MT, BN = 32 * NT;
    static constexpr int U = TYPE == 12 ? 9 : 13;       // 16-byte chunks per weight block
    static constexpr int XP = BM * 8 + 32;              // dwords per residue plane of x (padded: two planes' writes share no bank)
    struct Stage {
        uint32_t x[8 * XP];        // [residue][row][sub-block]: four int8, sign bit flipped
        uint32_t w[4 * U * BN];    // [dword][row]
        float xd[BM];
        uint32_t bs[TYPE == 12 ? BM * 8 : 4];  // [row][16] fp16 sums of 16
        float wd[BN];              // Q6_K
    };
    union {
        Stage st[2];
        float red[9 * 16 * 64];
    };
};

template <int TYPE, int MT, int NT>
__global__ __launch_bounds__(kMmThreads) void kq_mm_kernel(const uint8_t* __restrict__ w, const uint8_t* __restrict__ act, const uint32_t* __restrict__ xt,
                                                           float* __restrict__ y, const float* __restrict__ resid, int64_t M, int64_t N, int K, int64_t ldy,
                                                           int tiles_m, int tiles_n) {
    using Sh = KqMmShared<TYPE, MT, NT>;
    constexpr int BM = Sh::BM, BN = Sh::BN, U = Sh::U, XP = Sh::XP;
    extern __shared__ __align__(16) uint8_t smem_mm[];
    Sh& sh = *reinterpret_cast<Sh*>(smem_mm);
    // workgroups go to the XCDs round robin: the row tiles of one weight tile
    // take indices equal mod 8, so its weights are fetched into one L2
    const int q8 = blockIdx.x / 8;
    const int tn = (q8 / tiles_m) * 8 + blockIdx.x % 8, tm = q8 % tiles_m;
    if (tn >= tiles_n) return;
    const int tid = threadIdx.x, lane = tid & 63, l = __builtin_amdgcn_readfirstlane(tid >> 6), c32 = lane & 31, h = lane >> 5;
    const int nb = K >> 8;
    const int64_t m0 = int64_t(tm) * BM, n0 = int64_t(tn) * BN;
    // Q4_K's 6-bit scales (mins) of sub-blocks 4h .. 4h + 3: h = 0 the low six
    // bits of header dword 1 (2), h = 1 four bits of dword 3 under their top two
    // a constant in a vector register: and-or of a mask and the fp16 1024 bits
    // is then one instruction (its literal form takes two)
    auto in_vgpr = [](uint32_t v) {
        asm volatile("" : "+v"(v));
        return v;
    };
    const uint32_t magic = 0x64006400u, lom = in_vgpr(0x000F000Fu), him = in_vgpr(0x00F000F0u);
    uint32_t h2m[4];
    if constexpr (TYPE == 14) {
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) h2m[jj] = in_vgpr(0x00030003u << (2 * jj));
    }
    const uint32_t hs2 = h ? 2u : 0u, hm6 = h ? 0x30303030u : 0x3F3F3F3Fu, hm4 = h ? 0x0F0F0F0Fu : 0u;

    // ---- staging: this thread's chunks of a super-block
    constexpr int XC = BM * 16, WC = BN * U;  // 16-byte chunks of x and of the weights
    constexpr int XI = (XC + kMmThreads - 1) / kMmThreads, WI = (WC + kMmThreads - 1) / kMmThreads;
    const int R = kq_rows_per_tile(K), wpt = kq_waves_per_tile(K);
    // chunk indices fit 32 bits: kq_form() looks at the weights, the launcher slices the activation rows
    uint32_t xrow[XI];   // chunk tid % 16 of the row, super-block 0
    uint32_t wslot[WI];  // slot of super-block 0 of the chunk's row
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int idx = tid + i * kMmThreads;
        xrow[i] = uint32_t(min<int64_t>(m0 + (idx / 16) % BM, M - 1) * nb * 16 + idx % 16);
    }
#pragma unroll
    for (int i = 0; i < WI; ++i) {
        const int64_t n = min<int64_t>(n0 + (tid + i * kMmThreads) % BN, N - 1);
        wslot[i] = uint32_t(n / R * wpt * 64 + n % R);
    }
    const uint4* w4 = reinterpret_cast<const uint4*>(w);
    const uint4* x4 = reinterpret_cast<const uint4*>(xt);
    const uint16_t* dplane = reinterpret_cast<const uint16_t*>(w4 + kq_slots(N, K) * U);  // Q6_K
    // threads 0 .. BM-1: a row's scale; BM .. 3 BM - 1 (Q4_K): half of a row's sums of 16; Q6_K: the last BN the weight scales
    const int arow = tid < BM ? tid : (tid - BM) / 2;
    const uint8_t* ablk = act + min<int64_t>(m0 + (arow % BM), M - 1) * nb * kQ8KBytes;
    uint4 px[XI], pw[WI], pb;
    float pd;
    uint16_t ph;
    auto load = [&](int b) {
#pragma unroll
        for (int i = 0; i < XI; ++i)
            if (XC % kMmThreads == 0 || tid + i * kMmThreads < XC) px[i] = x4[xrow[i] + uint32_t(b) * 16];
#pragma unroll
        for (int i = 0; i < WI; ++i)
            if (tid + i * kMmThreads < WC) pw[i] = w4[mm_chunk_index(wslot[i] + uint32_t(b * R), (tid + i * kMmThreads) / BN, U)];
        if (tid < BM) {
            pd = *reinterpret_cast<const float*>(ablk + int64_t(b) * kQ8KBytes);
        } else if (TYPE == 12 && tid < 3 * BM) {
            const uint32_t* s = reinterpret_cast<const uint32_t*>(ablk + int64_t(b) * kQ8KBytes + 260) + 4 * ((tid - BM) & 1);
            pb = make_uint4(s[0], s[1], s[2], s[3]);
        } else if (TYPE == 14 && tid >= kMmThreads - BN) {
            ph = dplane[wslot[0] + uint32_t(b * R)];  // row tid % BN
        }
    };
    auto store = [&](typename Sh::Stage& st) {
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            const int idx = tid + i * kMmThreads;
            if (XC % kMmThreads == 0 || idx < XC) {
                // chunk c of a row: sub-block c / 2, residues 4 (c % 2) .. + 3
                uint32_t* dst = st.x + (4 * (idx & 1)) * XP + (idx / 16) * 8 + (idx % 16) / 2;
                dst[0] = px[i].x ^ 0x80808080u;
                dst[XP] = px[i].y ^ 0x80808080u;
                dst[2 * XP] = px[i].z ^ 0x80808080u;
                dst[3 * XP] = px[i].w ^ 0x80808080u;
            }
        }
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            const int idx = tid + i * kMmThreads;
            if (idx < WC) {
                uint32_t* dst = st.w + 4 * (idx / BN) * BN + idx % BN;
                dst[0] = pw[i].x;
                dst[BN] = pw[i].y;
                dst[2 * BN] = pw[i].z;
                dst[3 * BN] = pw[i].w;
            }
        }
        if (tid < BM) {
            st.xd[tid] = pd;
        } else if (TYPE == 12 && tid < 3 * BM) {
            auto two = [](uint32_t v) { return as_u32(h2_t{_Float16(int16_t(v & 0xFFFF)), _Float16(int16_t(v >> 16))}); };
            reinterpret_cast<uint4*>(st.bs)[tid - BM] = make_uint4(two(pb.x), two(pb.y), two(pb.z), two(pb.w));
        } else if (TYPE == 14 && tid >= kMmThreads - BN) {
            st.wd[tid - (kMmThreads - BN)] = half_bits_to_f32(ph);
        }
    };

    float acc[MT][NT][16], macc[16];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) macc[v] = 0.f;

    load(0);
    store(sh.st[0]);
    if (nb > 1) load(1);
    __syncthreads();
    constexpr int F = TYPE == 12 ? 2 : 4;  // MFMA operands per 32 weight rows
    // the weights of residue l, sub-blocks 4h .. 4h + 3, scaled
    auto weights = [&](const typename Sh::Stage& st, int j, h8_t (&wf)[F], float& wd) {
        const uint32_t* wr = st.w + 32 * j + c32;
        if constexpr (TYPE == 12) {
            wd = half_bits_to_f32(uint16_t(wr[0]));
            const uint32_t h1 = wr[BN], h3 = wr[3 * BN];
            const uint32_t sc = ((h1 >> hs2) & hm6) | (h3 & hm4);
#pragma unroll
            for (int c = 0; c < 2; ++c) {  // sub-blocks 2c (low nibbles) and 2c + 1 of the four
                const uint32_t g = wr[(4 + 8 * (2 * h + c) + l) * BN], g8 = g >> 8;
                const h2_t s0 = byte_twice(sc, 2 * c) - h2_of(1024.f), s1 = (byte_twice(sc, 2 * c + 1) - h2_of(1024.f)) * h2_of(0.0625f);
                const h2_t a0 = s0 * h2_of(-1024.f), a1 = s1 * h2_of(-1024.f);
                // (1024 + q) s - 1024 s and (1024 + 16 q) s / 16 - 64 s: exact, one rounding each
                wf[c] = h8_of(h2_fma(as_h2((g & lom) | magic), s0, a0), h2_fma(as_h2((g & him) | magic), s1, a1),
                              h2_fma(as_h2((g8 & lom) | magic), s0, a0), h2_fma(as_h2((g8 & him) | magic), s1, a1));
            }
        } else {
            wd = st.wd[32 * j + c32];
            const uint32_t qh = wr[(32 + 8 * h + l) * BN], qh8 = qh >> 8;
#pragma unroll
            for (int c = 0; c < 2; ++c) {  // sub-blocks c (low nibbles) and c + 2 of the four
                const uint32_t g = wr[(8 * (2 * h + c) + l) * BN], g8 = g >> 8;
                h2_t lo[4], hi[4];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int jj = c + 2 * t;
                    // scales of the sub-block's halves (i = 0, 1 | 2, 3), int8
                    const uint32_t sw = wr[(48 + 2 * h + jj / 2) * BN] ^ 0x80808080u;
                    const h2_t s = as_h2(__builtin_amdgcn_perm(0x64646464u, sw, jj % 2 ? 0x04030402u : 0x04010400u)) - h2_of(1152.f);
                    // low bits: lo4 s / 16 from 1024 + lo4 (or 1024 + 16 lo4)
                    const h2_t ls = s * h2_of(t ? 0.00390625f : 0.0625f), la = s * h2_of(t ? -4.f : -64.f);
                    const uint32_t lm = t ? him : lom;
                    lo[t] = h2_fma(as_h2((g & lm) | magic), ls, la);
                    lo[2 + t] = h2_fma(as_h2((g8 & lm) | magic), ls, la);
                    // high bits, at 2 jj of each byte: (hi2 - 2) s
                    const uint32_t hm = h2m[jj];
                    const h2_t hs = s * h2_of(1.f / float(1 << (2 * jj))), hb = h2_of(-1024.f - float(2 << (2 * jj)));
                    hi[t] = (as_h2((qh & hm) | magic) + hb) * hs;
                    hi[2 + t] = (as_h2((qh8 & hm) | magic) + hb) * hs;
                }
                wf[2 * c] = h8_of(lo[0], lo[1], lo[2], lo[3]);
                wf[2 * c + 1] = h8_of(hi[0], hi[1], hi[2], hi[3]);
            }
        }
    };
    // the activations of residue l, sub-blocks 4h .. 4h + 3 (Q6_K: times 16)
    auto activations = [&](const typename Sh::Stage& st, h8_t (&xf)[MT][2], float& xd) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const uint4 xv = *reinterpret_cast<const uint4*>(st.x + l * XP + (32 * i + c32) * 8 + 4 * h);
            auto cv = [](h2_t t) {
                if constexpr (TYPE == 12) return t - h2_of(1152.f);
                return h2_fma(t, h2_of(16.f), h2_of(-18432.f));
            };
            const uint32_t a0 = xv.x, a1 = TYPE == 12 ? xv.y : xv.z, b0 = TYPE == 12 ? xv.z : xv.y, b1 = xv.w;
            xf[i][0] = h8_of(cv(bytes_even(a0)), cv(bytes_even(a1)), cv(bytes_odd(a0)), cv(bytes_odd(a1)));
            xf[i][1] = h8_of(cv(bytes_even(b0)), cv(bytes_even(b1)), cv(bytes_odd(b0)), cv(bytes_odd(b1)));
        }
        xd = st.xd[MT == 2 ? lane : c32];
    };
    auto products = [&](const h8_t (&xf)[MT][2], const h8_t (&wf)[F], f16v_t (&aux)[MT]) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            aux[i] = f16v_t{};
#pragma unroll
            for (int f = 0; f < F; ++f) aux[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[i][F == 2 ? f : f / 2], wf[f], aux[i], 0, 0, 0);
        }
    };
    auto chains = [&](int j, float xd, float wd, const f16v_t (&aux)[MT]) {
        const f32v_t d = __builtin_amdgcn_mfma_f32_32x32x1f32(xd, wd, f32v_t{}, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                acc[i][j][v] += d[16 * i + v] * aux[i][v];
                asm volatile("" : "+v"(acc[i][j][v]));  // here, not sunk past what follows with d and aux kept
            }
        }
    };
    // One super-block's last chains run beside the next one's decoding, and its
    // later products beside its first chains: the eight waves meet at a barrier
    // per super-block, so what one wave does not overlap nothing does.
    h8_t xf[MT][2], wf[F];
    float xd, wd;
    activations(sh.st[0], xf, xd);
    weights(sh.st[0], 0, wf, wd);
    for (int b = 0; b < nb; ++b) {
        const auto& st = sh.st[b & 1];
        const auto& nx = sh.st[(b + 1) & 1];
        f16v_t aux[NT][MT];
        // the other buffer's readers finished at the last barrier
        if (b + 1 < nb) store(sh.st[(b + 1) & 1]);
        if (b + 2 < nb) load(b + 2);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (TYPE == 12) {
            if (l < MT * NT) {  // the mins term of tile l
                const int i = l % MT, j = l / MT;
                const uint32_t* wr = st.w + 32 * j + c32;
                const uint32_t h2 = wr[2 * BN], h3 = wr[3 * BN];
                const float wdm = half_bits_to_f32(uint16_t(wr[0] >> 16)), xdm = st.xd[32 * i + c32];
                const uint32_t mn = ((h2 >> hs2) & hm6) | ((h3 >> 4) & hm4);
                const h8_t mf = h8_of(byte_twice(mn, 0) - h2_of(1024.f), byte_twice(mn, 1) - h2_of(1024.f), byte_twice(mn, 2) - h2_of(1024.f),
                                      byte_twice(mn, 3) - h2_of(1024.f));
                const h8_t bf = __builtin_bit_cast(h8_t, reinterpret_cast<const uint4*>(st.bs)[(32 * i + c32) * 2 + h]);
                const f16v_t sumi = __builtin_amdgcn_mfma_f32_32x32x16_f16(bf, mf, f16v_t{}, 0, 0, 0);
                // one product per output: the second of the two terms is 0 * 0
                const f16v_t dm = __builtin_amdgcn_mfma_f32_32x32x2f32(h ? 0.f : xdm, h ? 0.f : wdm, f16v_t{}, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    macc[v] -= dm[v] * sumi[v];
                    asm volatile("" : "+v"(macc[v]));
                }
            }
        }
        products(xf, wf, aux[0]);
        if constexpr (NT == 2) {
            h8_t wf1[F];
            float wd1;
            weights(st, 1, wf1, wd1);
            __builtin_amdgcn_sched_barrier(0);
            products(xf, wf1, aux[1]);
            chains(0, xd, wd, aux[0]);
            wd = wd1;
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        const float xdl = xd, wdl = wd;
        activations(nx, xf, xd);  // past the last super-block: stale words, not used
        weights(nx, 0, wf, wd);
        chains(NT - 1, xdl, wdl, aux[NT - 1]);
    }

    // sumf = mins chain, then += sums[0..7]
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
#pragma unroll
            for (int v = 0; v < 16; ++v) sh.red[(l * 16 + v) * 64 + lane] = acc[i][j][v];
            if (TYPE == 12 && l == j * MT + i) {
#pragma unroll
                for (int v = 0; v < 16; ++v) sh.red[(128 + v) * 64 + lane] = macc[v];
            }
            __syncthreads();
#pragma unroll
            for (int e = tid; e < 1024; e += kMmThreads) {
                float sumf = TYPE == 12 ? sh.red[8 * 1024 + e] : 0.f;
#pragma unroll
                for (int p = 0; p < 8; ++p) sumf += sh.red[p * 1024 + e];
                const int v = e >> 6, el = e & 63;
                const int64_t m = m0 + 32 * i + 8 * (v / 4) + 4 * (el >> 5) + v % 4, n = n0 + 32 * j + (el & 31);
                if (m < M && n < N) {
                    const int64_t o = m * ldy + n;
                    y[o] = resid ? resid[o] + sumf : sumf;
                }
            }
            __syncthreads();
        }
    }
}

// Q5_K against fp32 activations (no integer-activation kernel in the
// reference): per block the dequant-in-dot chain of nm/src/quant.hpp:207-229
// -- acc += (d1 * q - m1) * x, 256 products in order from acc = 0 -- and per
// output the sum of its blocks' results in order (quant_i8.hpp:403-407).
// Lane (b, r) keeps its 176-byte block in registers; TILE activation rows at a
// time are staged in shared memory and each weight is decoded once for all of
// them. grid (ceil(N / R), ceil(M / rows_per_group)).
template <int TILE>
__global__ __launch_bounds__(kKqThreads) void q5k_gemm_kernel(const uint8_t* __restrict__ w, const float* __restrict__ x, int64_t ldx, float* __restrict__ y,
                                                              const float* __restrict__ resid, int64_t M, int64_t N, int K, int64_t ldy, int R,
                                                              int rows_per_group) {
    // x position-major [K][TILE] (the TILE rows' values of one position are
    // adjacent: one read, constant offsets from the lane's block); once every
    // lane has its results the same memory holds the block results
    // [TILE][R * nb] (R * nb <= 256 <= K)
    extern __shared__ __align__(16) float smem[];
    float* xs = smem;
    float* res = smem;
    const int nb = K >> 8, tid = threadIdx.x, items = R * nb;
    const int64_t n0 = int64_t(blockIdx.x) * R;
    const int64_t m_begin = int64_t(blockIdx.y) * rows_per_group;
    const int64_t m_end = min(M, m_begin + rows_per_group);
    const int b = tid / R, r = tid % R;
    const bool active = tid < items && n0 + r < N;

    uint32_t qh[8], qs[32];
    float d1[8], m1[8];
    if (active) {
        const int64_t slot = (int64_t(blockIdx.x) * ((items + 63) / 64) + tid / 64) * 64 + tid % 64;
        const uint4* src = reinterpret_cast<const uint4*>(w) + kq_chunk_index(slot, 0, 11);  // chunk u at src[64 u]
        const uint4 hdr = src[0];
        const uint8_t* hb = reinterpret_cast<const uint8_t*>(&hdr);
        const float d = half_bits_to_f32(uint16_t(hdr.x & 0xFFFF)), dmin = half_bits_to_f32(uint16_t(hdr.x >> 16));
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            int sc, m;
            scale_min_k4(hb + 4, j, sc, m);
            d1[j] = d * float(sc);
            m1[j] = dmin * float(m);
        }
        const uint4 h0 = src[64], h1 = src[128];
        qh[0] = h0.x, qh[1] = h0.y, qh[2] = h0.z, qh[3] = h0.w, qh[4] = h1.x, qh[5] = h1.y, qh[6] = h1.z, qh[7] = h1.w;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint4 v = src[64 * (3 + i)];
            qs[4 * i] = v.x, qs[4 * i + 1] = v.y, qs[4 * i + 2] = v.z, qs[4 * i + 3] = v.w;
        }
    }

    for (int64_t mt = m_begin; mt < m_end; mt += TILE) {
        const int mrows = int(min<int64_t>(TILE, m_end - mt));
        for (int i = tid; i < TILE * (K >> 2); i += kKqThreads) {
            const int mi = i / (K >> 2), c4 = i % (K >> 2);
            const float4 v = mi < mrows ? reinterpret_cast<const float4*>(x + (mt + mi) * ldx)[c4] : make_float4(0.f, 0.f, 0.f, 0.f);
            xs[(4 * c4) * TILE + mi] = v.x;
            xs[(4 * c4 + 1) * TILE + mi] = v.y;
            xs[(4 * c4 + 2) * TILE + mi] = v.z;
            xs[(4 * c4 + 3) * TILE + mi] = v.w;
        }
        __syncthreads();
        float acc[TILE];
#pragma unroll
        for (int mi = 0; mi < TILE; ++mi) acc[mi] = 0.f;
        if (active) {
            const float* xb = xs + 256 * TILE * b;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int j = 2 * c + h;
#pragma unroll
                    for (int i4 = 0; i4 < 8; ++i4) {  // 4 weights: bytes 4 i4 .. 4 i4 + 3 of the 32
                        // opaque copies: decoded per pass instead of 256 decoded
                        // weights hoisted out of the row loop into registers
                        uint32_t qw = qs[8 * c + i4], fifth = qh[i4];
                        asm volatile("" : "+v"(qw), "+v"(fifth) : : "memory");
                        // byte u = the 4-bit value + 16 * its fifth bit (bit j of
                        // byte u of qh): four 5-bit weights in one dword, each
                        // converted by a byte-to-float conversion
                        const uint32_t q5 = ((qw >> (4 * h)) & 0x0F0F0F0Fu) | (((fifth >> j) & 0x01010101u) << 4);
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const float wv = d1[j] * float((q5 >> (8 * u)) & 0xFFu) - m1[j];
                            const float* xp = xb + (64 * c + 32 * h + 4 * i4 + u) * TILE;
#pragma unroll
                            for (int mi = 0; mi < TILE; ++mi) acc[mi] += wv * xp[mi];
                        }
                        // the chains advance group by group (not deferred behind
                        // every group's decoded weights and reads)
#pragma unroll
                        for (int mi = 0; mi < TILE; ++mi) asm volatile("" : "+v"(acc[mi]));
                    }
                }
            }
        }
        __syncthreads();  // every lane's reads of xs are done
        if (active) {
#pragma unroll
            for (int mi = 0; mi < TILE; ++mi)
                if (mi < mrows) res[mi * items + tid] = acc[mi];
        }
        __syncthreads();
        for (int idx = tid; idx < mrows * R; idx += kKqThreads) {
            const int mi = idx / R, rr = idx % R;
            const int64_t n = n0 + rr;
            if (n >= N) continue;
            float s = 0.f;
            for (int bb = 0; bb < nb; ++bb) s += res[mi * items + bb * R + rr];
            const int64_t o = (mt + mi) * ldy + n;
            y[o] = resid ? resid[o] + s : s;
        }
        __syncthreads();
    }
}

// ---- Q5_K products of several activation rows ---------------------------------------------
// The reference rounds each product wv * x and then each sum, 256 in order per
// super-block, so nothing can be contracted; the work is one multiply and one
// add per weight and row. The multiplies of a position's R rows x 64 weight
// rows come as one fp32 MFMA of depth 1 (an outer product with a zero addend:
// every entry the correctly rounded product), which needs one value of x and
// one weight per lane where vector multiplies would need every row's x
// broadcast to each lane; the adds are vector instructions. Lane n decodes the
// weights of row n once for the R rows.
//
// A workgroup owns R activation rows x 64 weight rows; its eight waves take
// super-blocks w, w + 8, ... each with its 256-term chains in registers, and
// after every eight super-blocks one lane per output adds their results in
// order. Each wave stages its own x, 64 positions at a time, in shared memory
// (rows padded: 16 rows' 16-byte reads share no bank); no other wave reads it.
//
// Bound: the fp32 MFMA runs on the vector units, so a position of 16 rows costs
// a SIMD 34 clocks of products, 36 of adds and ~15 of decoding. Measured: 256
// rows x 4096, K 4096 506 -> 173 us, of which the multiplies and adds alone are
// 134 (before: every lane decoding its block per 4 rows, x from shared memory).
template <int R>
struct OuterF32;
template <>
struct OuterF32<4> {
    using V = float __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ V mul(float x, float w) { return __builtin_amdgcn_mfma_f32_4x4x1f32(x, w, V{}, 0, 0, 0); }
    static __device__ __forceinline__ int row(int v, int) { return v; }
    static __device__ __forceinline__ int col(int, int lane) { return lane; }
};
template <>
struct OuterF32<16> {
    using V = float __attribute__((ext_vector_type(16)));
    static __device__ __forceinline__ V mul(float x, float w) { return __builtin_amdgcn_mfma_f32_16x16x1f32(x, w, V{}, 0, 0, 0); }
    static __device__ __forceinline__ int row(int v, int lane) { return 4 * (lane >> 4) + (v & 3); }
    static __device__ __forceinline__ int col(int v, int lane) { return 16 * (v >> 2) + (lane & 15); }
};
constexpr int kQ5Waves = 8;
constexpr int kQ5Pos = 64;             // positions staged at a time
constexpr int kQ5Ld = kQ5Pos + 4;      // padded row
constexpr size_t q5k_mm_shared(int R) { return size_t(kQ5Waves) * R * kQ5Ld * 4; }

template <int R>
__global__ __launch_bounds__(64 * kQ5Waves) void q5k_mm_kernel(const uint8_t* __restrict__ w, const float* __restrict__ x, int64_t ldx, float* __restrict__ y,
                                                               const float* __restrict__ resid, int64_t M, int64_t N, int K, int64_t ldy) {
    using Outer = OuterF32<R>;
    using V = typename Outer::V;
    extern __shared__ __align__(16) float smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nb = K >> 8;
    const int64_t n0 = int64_t(blockIdx.x) * 64, m0 = int64_t(blockIdx.y) * R;
    float* xs = smem + wave * R * kQ5Ld;
    const int64_t n = min<int64_t>(n0 + lane, N - 1);
    const int rows_per_tile = kq_rows_per_tile(K);
    const int64_t slot0 = n / rows_per_tile * kq_waves_per_tile(K) * 64 + n % rows_per_tile;

    // staging of 64 positions of R rows: 16 lanes per row
    constexpr int XI = R / 4;
    const float* xrow[XI];
#pragma unroll
    for (int i = 0; i < XI; ++i) xrow[i] = x + min<int64_t>(m0 + 4 * i + lane / 16, M - 1) * ldx + 4 * (lane % 16);
    float4 px[XI];
    auto load = [&](int k) {
#pragma unroll
        for (int i = 0; i < XI; ++i) px[i] = *reinterpret_cast<const float4*>(xrow[i] + k);
    };

    constexpr int OUT = R * 64 / (64 * kQ5Waves) > 0 ? R * 64 / (64 * kQ5Waves) : 1;
    float sum[OUT];
#pragma unroll
    for (int i = 0; i < OUT; ++i) sum[i] = 0.f;

    for (int b0 = 0; b0 < nb; b0 += kQ5Waves) {
        const int b = b0 + wave;
        if (b < nb) {
            load(256 * b);
            const int64_t slot = slot0 + int64_t(b) * rows_per_tile;
            const uint4* src = reinterpret_cast<const uint4*>(w) + kq_chunk_index(slot, 0, 11);  // chunk u at src[64 u]
            const uint4 hdr = src[0], h0 = src[64], h1 = src[128];
            // the 6-bit scales and mins of sub-blocks 0..3 and 4..7, a byte each
            const uint32_t sc4[2] = {hdr.y & 0x3F3F3F3Fu, (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u)};
            const uint32_t mn4[2] = {hdr.z & 0x3F3F3F3Fu, ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u)};
            const float d = half_bits_to_f32(uint16_t(hdr.x & 0xFFFF)), dmin = half_bits_to_f32(uint16_t(hdr.x >> 16));
            uint32_t qh[8] = {h0.x, h0.y, h0.z, h0.w, h1.x, h1.y, h1.z, h1.w};
            uint4 q0 = src[64 * 3], q1 = src[64 * 4];
            V acc{}, prod{};  // prod: the products of the position before, added while the next ones form
#pragma unroll 1
            for (int c = 0; c < 4; ++c) {
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int i = 0; i < XI; ++i) *reinterpret_cast<float4*>(xs + (4 * i + lane / 16) * kQ5Ld + 4 * (lane % 16)) = px[i];
                __builtin_amdgcn_wave_barrier();
                const uint32_t qs[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
                if (c < 3) {
                    load(256 * b + kQ5Pos * (c + 1));
                    q0 = src[64 * (3 + 2 * (c + 1))], q1 = src[64 * (4 + 2 * (c + 1))];
                }
                __builtin_amdgcn_sched_barrier(0);
                const float* xl = xs + (lane % R) * kQ5Ld;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int j = 2 * c + h;
                    const float d1 = d * float((sc4[c >> 1] >> (8 * (j & 3))) & 0xFFu), m1 = dmin * float((mn4[c >> 1] >> (8 * (j & 3))) & 0xFFu);
#pragma unroll
                    for (int i4 = 0; i4 < 8; ++i4) {
                        const float4 xv = *reinterpret_cast<const float4*>(xl + 32 * h + 4 * i4);
                        // byte u = the 4-bit value + 16 * its fifth bit (bit j of byte u of qh)
                        const uint32_t q5 = ((qs[i4] >> (4 * h)) & 0x0F0F0F0Fu) | (((qh[i4] >> j) & 0x01010101u) << 4);
                        const float xe[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const float wv = d1 * float((q5 >> (8 * u)) & 0xFFu) - m1;
                            const V next = Outer::mul(xe[u], wv);
                            acc += prod;
                            prod = next;
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
            }
            acc += prod;
            __builtin_amdgcn_wave_barrier();
            float* res = xs;  // [R][64]
#pragma unroll
            for (int v = 0; v < R; ++v) res[Outer::row(v, lane) * 64 + Outer::col(v, lane)] = acc[v];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < OUT; ++i) {
            const int e = tid + 64 * kQ5Waves * i;
            if (e < R * 64)
                for (int p = 0; p < min(kQ5Waves, nb - b0); ++p) sum[i] += smem[p * R * kQ5Ld + e];
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < OUT; ++i) {
        const int e = tid + 64 * kQ5Waves * i;
        const int64_t m = m0 + e / 64, nn = n0 + e % 64;
        if (e < R * 64 && m < M && nn < N) {
            const int64_t o = m * ldy + nn;
            y[o] = resid ? resid[o] + sum[i] : sum[i];
        }
    }
}

// GGUF -> packed K-quant layout. Within a block: Q4_K keeps its 16-byte
// header; its 128 quant bytes become 32 residue dwords: dword 8c + l, byte i =
// qs[32c + 8i + l] (low nibbles: sub-block 2c, high: 2c + 1). Q6_K's 128 ql
// bytes take the same permutation (pair c = sub-blocks {j, j + 2} of half
// c / 2), its 64 qh bytes too (dword 8h + l, byte i = qh[32h + 8i + l]: 2-bit
// fields of sub-blocks 4h .. 4h + 3), then the 16 scales; its d goes to the d
// plane. Q5_K keeps its bytes. The blocks then take the slots of the tiled
// structure-of-arrays layout above. One lane per output dword of a block.
__global__ __launch_bounds__(256) void kq_pack_kernel(int type, const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, int64_t N, int64_t K) {
    const int nb = int(K / 256), U = kq_chunks(type), words = 4 * U + 1;  // + the Q6_K d
    const int64_t gid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (gid >= N * nb * words) return;
    const int64_t f = gid / words;  // GGUF block: row f / nb, block f % nb
    const int wi = int(gid % words);
    const int64_t slot = kq_slot(f / nb, int(f % nb), K);
    const int bytes = type == 12 ? 144 : type == 13 ? 176 : 210;
    const uint8_t* s = src + f * bytes;
    if (wi == 4 * U) {  // Q6_K d
        if (type == 14) reinterpret_cast<uint16_t*>(dst + kq_slots(N, K) * 13 * 16)[slot] = uint16_t(s[208] | (s[209] << 8));
        return;
    }
    const uint8_t* g;   // the dword's four source bytes: g[0], g[step], g[2 step], g[3 step]
    int step = 1;
    if (type == 13) {
        g = s + 4 * wi;
    } else if (type == 12) {
        if (wi < 4) {
            g = s + 4 * wi;
        } else {
            const int dw = wi - 4;
            g = s + 16 + 32 * (dw / 8) + dw % 8;
            step = 8;
        }
    } else if (wi < 32) {
        g = s + 32 * (wi / 8) + wi % 8;
        step = 8;
    } else if (wi < 48) {
        const int dw = wi - 32;
        g = s + 128 + 32 * (dw / 8) + dw % 8;
        step = 8;
    } else {
        g = s + 192 + 4 * (wi - 48);
    }
    const uint32_t v = uint32_t(g[0]) | (uint32_t(g[step]) << 8) | (uint32_t(g[2 * step]) << 16) | (uint32_t(g[3 * step]) << 24);
    reinterpret_cast<uint32_t*>(dst)[kq_chunk_index(slot, wi / 4, U) * 4 + wi % 4] = v;
}

// Weight::dequant_row (nm/src/quant.hpp:322-395) of the rows `ids` of a
// packed Q4_K / Q6_K or GGUF Q5_K tensor: Q4_K / Q5_K d1 * q - m1 with
// d1 = d * sc, m1 = dmin * m; Q6_K (d * sc) * (q - 32). grid (nb, n_ids), 256 lanes.
__global__ __launch_bounds__(256) void kq_dequant_rows_kernel(int type, const uint8_t* __restrict__ w, int64_t N, int K, const int32_t* __restrict__ ids,
                                                              float* __restrict__ out) {
    const int b = blockIdx.x, p = threadIdx.x;
    const int64_t t = blockIdx.y;
    const int32_t id = ids[t];
    float* o = out + t * K + 256 * b + p;
    if (id < 0 || id >= N) {  // the host validates ids; a bad one gives zeros, never a stray read
        *o = 0.f;
        return;
    }
    const int64_t slot = kq_slot(id, b, K);
    const int U = kq_chunks(type);
    // byte o of the block in `slot`
    auto at = [&](int o) { return w[kq_chunk_index(slot, o >> 4, U) * 16 + (o & 15)]; };
    const int j = p >> 5, i = (p & 31) >> 3, l = p & 7;
    if (type == 12 || type == 13) {
        uint8_t hdr[16];
#pragma unroll
        for (int o = 0; o < 16; ++o) hdr[o] = at(o);
        const uint8_t* s = hdr;
        const float d = half_bits_to_f32(uint16_t(s[0] | (s[1] << 8))), dmin = half_bits_to_f32(uint16_t(s[2] | (s[3] << 8)));
        int sc, m;
        scale_min_k4(s + 4, j, sc, m);
        const float dd = d * float(sc), mm = dmin * float(m);
        int q;
        if (type == 12) {
            q = (at(16 + 4 * (8 * (j >> 1) + l) + i) >> (4 * (j & 1))) & 0xF;
        } else {
            const int e = p & 31;
            q = ((at(48 + 32 * (j >> 1) + e) >> (4 * (j & 1))) & 0xF) + (((at(16 + e) >> j) & 1) << 4);
        }
        *o = dd * float(q) - mm;
        return;
    }
    const int cp = 2 * (j >> 2) + (j & 1);
    const int lo = (at(4 * (8 * cp + l) + i) >> (4 * ((j & 3) >> 1))) & 0xF;
    const int hi = (at(128 + 4 * (8 * (j >> 2) + l) + i) >> (2 * (j & 3))) & 3;
    const float d = half_bits_to_f32(reinterpret_cast<const uint16_t*>(w + kq_slots(N, K) * 13 * 16)[slot]);
    const int sc = int(int8_t(at(192 + (p >> 4))));
    *o = d * float(sc) * float((lo | (hi << 4)) - 32);
}

}  // namespace

// GGUF Q8_K blocks, then (16-byte aligned) the regrouped int8 copy: 256 bytes per block
int64_t act_q8_K_bytes(int64_t m, int64_t k) { return ((m * (k / 256) * kQ8KBytes + 15) & ~int64_t(15)) + m * (k / 256) * 256; }

static const uint32_t* regrouped_of(const void* act, int64_t nblocks) {
    return reinterpret_cast<const uint32_t*>(static_cast<const uint8_t*>(act) + ((nblocks * kQ8KBytes + 15) & ~int64_t(15)));
}

void launch_quantize_q8_K(const float* x, void* act, int64_t M, int64_t K, hipStream_t s) {
    const int64_t nblocks = M * (K / 256);
    auto* xt = const_cast<uint32_t*>(regrouped_of(act, nblocks));
    hipLaunchKernelGGL(quantize_q8_K_kernel, dim3(unsigned(nblocks)), dim3(64), 0, s, x, static_cast<uint8_t*>(act), xt, nblocks);
}

int64_t kquant_packed_bytes(int type, int64_t N, int64_t K) {
    const int64_t slots = kq_slots(N, K);
    return slots * kq_chunks(type) * 16 + (type == 14 ? slots * 2 : 0);
}

void launch_kquant_pack(int type, const void* gguf, void* packed, int64_t N, int64_t K, hipStream_t s) {
    // the padding slots stay zero (never read)
    hip_check(hipMemsetAsync(packed, 0, size_t(kquant_packed_bytes(type, N, K)), s), "pack clear");
    const int64_t work = N * (K / 256) * (4 * kq_chunks(type) + 1);
    hipLaunchKernelGGL(kq_pack_kernel, dim3(unsigned((work + 255) / 256)), dim3(256), 0, s, type, static_cast<const uint8_t*>(gguf),
                       static_cast<uint8_t*>(packed), N, K);
}

// rows per workgroup (R) and activation rows per workgroup for an (M, N, K)
// product: R * nb <= 256 lanes; rows split over grid.y while that leaves at
// least ~2048 workgroups
static void kq_plan(int64_t M, int64_t N, int64_t K, int tile, int* R, int* rows_per_group) {
    *R = kq_rows_per_tile(K);  // the packed layout's tile
    const int64_t gx = (N + *R - 1) / *R;
    const int64_t want_y = std::max<int64_t>(1, (2048 + gx - 1) / gx);
    const int64_t gy = std::min<int64_t>(want_y, (M + tile - 1) / tile);
    int64_t per = (M + gy - 1) / gy;
    per = (per + tile - 1) / tile * tile;
    *rows_per_group = int(per);
}

int kquant_max_k(int type) { return type == 13 ? 16384 : 65536; }

template <int TYPE, int MT, int NT>
static void kq_mm(const uint8_t* w, const uint8_t* act, const uint32_t* xt, float* y, const float* resid, int64_t M, int64_t N, int64_t K, int64_t ldy,
                  hipStream_t s) {
    const int64_t tm = (M + 32 * MT - 1) / (32 * MT), tn = (N + 32 * NT - 1) / (32 * NT);
    const dim3 grid(unsigned((tn + 7) / 8 * 8 * tm));
    hipLaunchKernelGGL((kq_mm_kernel<TYPE, MT, NT>), grid, dim3(kMmThreads), sizeof(KqMmShared<TYPE, MT, NT>), s, w, act, xt, y, resid, M, N, int(K), ldy,
                       int(tm), int(tn));
}

// Activation rows of one launch of kq_mm_kernel: 2^20 for its 32-bit activation
// chunk indices, fewer where N is so large that the grid would pass 2^32 - 1
// lanes (0: not even one tile of rows fits).
constexpr int64_t kq_slice_rows(int64_t N, int64_t tile) {
    const int64_t columns = ((N + tile - 1) / tile + 7) / 8 * 8, workgroups = ((int64_t(1) << 32) - 1) / kMmThreads;
    return std::min(int64_t(1) << 20, workgroups / columns * tile);
}
static_assert(kq_slice_rows(32768 - 512, 64) == 1 << 20);  // 504 tile columns x 16384
static_assert(kq_slice_rows(32768, 64) == (1 << 20) - 64);  // 512 x 16384 workgroups of 512 lanes are 2^32
static_assert(kq_slice_rows((int64_t(1) << 32) / 9, 64) == 64 && kq_slice_rows(int64_t(1) << 28, 32) == 0);

// The form of a Q4_K / Q6_K product: 1 the lane-per-block form, 32 or 64 the
// matrix-core form with tiles of that many rows either way.
static int kq_form(int type, int64_t M, int64_t N, int64_t K) {
    // kq_mm_kernel's weight chunk indices are 32 bits; kq_gemm_kernel's are 64
    // (477M super-blocks of Q4_K, 330M of Q6_K: 69 GB)
    if (M == 1 || kq_slots(N, K) * kq_chunks(type) > int64_t(UINT32_MAX)) return 1;
    // Which form, by estimates in microseconds (with the quantizer, fitted to
    // M 2 .. 48, N 1000 .. 12288, K 1024 .. 12288): the lane-per-block form
    // costs per pass of R weight rows x 4 activation rows on a compute unit,
    // the matrix-core form per round of one 32 x 32 tile a compute unit (a
    // 64 x 64 tile costs two) and super-block. Measured, former and matrix-core
    // form: Q4_K 4096 x 4096: 12 rows 16.3 / 19.7, 16 rows 22.9 / 19.9, 48 rows
    // 44.8 / 20.8; 1000 x 12288, 16 rows 26.7 / 44.3; Q6_K 4096 x 4096: 8 rows
    // 18.2 / 19.4, 12 rows 27.2 / 21.6; 4096 x 12288, 9 rows 68.7 / 50.3.
    const int nb = int(K / 256);
    const int64_t cus = device_cus();
    auto rounds = [&](int64_t t) { return ((M + t - 1) / t * ((N + t - 1) / t) + cus - 1) / cus; };
    const int64_t small = rounds(32), large = rounds(64), R = kq_rows_per_tile(K);
    const double passes = double((N + R - 1) / R) * double(M) / (4.0 * double(cus)), over = std::max(0, nb - 32);
    const double lanes = type == 12 ? 9 + (3 + 0.1 * over) * passes : 10 + (5.2 + 0.06 * over) * passes;
    const double tiles = (6 + (type == 12 ? 0.83 : 0.92) * nb) * (0.23 + 0.77 * double(std::min(small, 2 * large)));
    if (tiles > lanes) return 1;
    // the small tile takes about half the large one's time for a quarter of its
    // outputs (Q4_K N 4096, K 4096: 64 rows 21 and 33 us, 509 rows 98 and 63 us)
    const int tile = small <= 2 * large ? 32 : 64;
    return kq_slice_rows(N, tile) > 0 ? tile : 1;
}

void launch_kquant_gemm_ld(int type, const void* w, const void* act, float* y, const float* resid, int64_t M, int64_t N, int64_t K, int64_t ldy,
                           hipStream_t s) {
    const int nb = int(K / 256);
    const auto* wb = static_cast<const uint8_t*>(w);
    const auto* ab = static_cast<const uint8_t*>(act);
    const uint32_t* xt = regrouped_of(act, M * nb);
    const int form = kq_form(type, M, N, K);
    if (form != 1) {
        auto run = form == 32 ? (type == 12 ? kq_mm<12, 1, 1> : kq_mm<14, 1, 1>) : (type == 12 ? kq_mm<12, 2, 2> : kq_mm<14, 2, 2>);
        const int64_t slice = kq_slice_rows(N, form);
        for (int64_t r0 = 0; r0 < M; r0 += slice)
            run(wb, ab + r0 * nb * kQ8KBytes, xt + r0 * nb * 64, y + r0 * ldy, resid ? resid + r0 * ldy : nullptr, std::min(slice, M - r0), N, K, ldy, s);
        return;
    }
    int R, per;
    kq_plan(M, N, K, kKqTile, &R, &per);
    const dim3 grid(unsigned((N + R - 1) / R), unsigned((M + per - 1) / per));
    if (type == 12) {
        const size_t lds = size_t(kKqTile) * R * nb * 9 * 4;
        auto kernel = M == 1 ? kq_gemm_kernel<12, true> : kq_gemm_kernel<12, false>;
        hipLaunchKernelGGL(kernel, grid, dim3(kKqThreads), lds, s, wb, ab, xt, y, resid, M, N, int(K), ldy, R, per);
    } else {
        const size_t lds = size_t(kKqTile) * R * nb * 8 * 4;
        auto kernel = M == 1 ? kq_gemm_kernel<14, true> : kq_gemm_kernel<14, false>;
        hipLaunchKernelGGL(kernel, grid, dim3(kKqThreads), lds, s, wb, ab, xt, y, resid, M, N, int(K), ldy, R, per);
    }
}

void launch_kquant_gemm(int type, const void* w, const void* act, float* y, int64_t M, int64_t N, int64_t K, hipStream_t s) {
    launch_kquant_gemm_ld(type, w, act, y, nullptr, M, N, K, N, s);
}

// activation rows per pass of the lane-per-block form: shared memory holds as many rows of K floats (<= 64 KiB)
static int q5k_tile(int64_t M, int64_t K) { return M == 1 ? 1 : K <= 4096 ? 4 : K <= 8192 ? 2 : 1; }

// The form of a Q5_K product: 1 the lane-per-block form, 4 or 16 the
// outer-product form with that many activation rows per tile.
static int q5k_form(int64_t M, int64_t N, int64_t K) {
    // Several rows: the outer-product form unless the lane-per-block form's
    // workgroup passes (one per R weight rows and tile activation rows; about 8,
    // 6.6 and 5 us each on a compute unit, at least 13) cost less than its 4-row
    // tiles (about 3 + 1.2 us per super-block of a row), both in microseconds.
    // Measured, former and this form: K 4096 x 4096 rows: 8 rows 19.4 / 22.1 us,
    // 10 rows 35.4 / 22.7; K 1024 x 1000, 2 rows: 12.8 / 9.4; K 8192 x 4096, 4
    // rows 27.3 / 39.8, 8 rows 53.2 / 41.1; K 12288 x 4096, 2 rows 45 / 62, 4 rows 80 / 61.
    if (M == 1) return 1;
    const int64_t cus = device_cus(), nb = K / 256;
    const int tile = q5k_tile(M, K);
    auto rounds = [&](int64_t rows, int64_t cols) { return ((M + rows - 1) / rows * ((N + cols - 1) / cols) + cus - 1) / cus; };
    const double lanes = std::max(13.0, double(rounds(tile, kq_rows_per_tile(K))) * (tile == 4 ? 8.0 : tile == 2 ? 6.6 : 5.0));
    if (double(rounds(4, 64)) * (3.0 + 1.2 * double(nb)) >= lanes) return 1;
    // 16-row tiles take three times a 4-row tile's time once the compute units
    // are full (47 and 15.5 us at K 4096)
    return 3 * rounds(16, 64) < rounds(4, 64) ? 16 : 4;
}

int kquant_gemm_plan(int type, int64_t M, int64_t N, int64_t K) { return type == 13 ? q5k_form(M, N, K) : kq_form(type, M, N, K); }

void launch_q5k_gemm(const void* w, const float* x, int64_t ldx, float* y, const float* resid, int64_t M, int64_t N, int64_t K, int64_t ldy, hipStream_t s) {
    const int rows = q5k_form(M, N, K);
    if (rows != 1) {
        const int64_t slice = int64_t(65535) * rows;  // grid.y
        for (int64_t r0 = 0; r0 < M; r0 += slice) {
            const int64_t part = std::min(slice, M - r0);
            hipLaunchKernelGGL(rows == 16 ? q5k_mm_kernel<16> : q5k_mm_kernel<4>, dim3(unsigned((N + 63) / 64), unsigned((part + rows - 1) / rows)),
                               dim3(64 * kQ5Waves), q5k_mm_shared(rows), s, static_cast<const uint8_t*>(w), x + r0 * ldx, ldx, y + r0 * ldy,
                               resid ? resid + r0 * ldy : nullptr, part, N, int(K), ldy);
        }
        return;
    }
    const int tile = q5k_tile(M, K);
    int R, per;
    kq_plan(M, N, K, tile, &R, &per);
    const dim3 grid(unsigned((N + R - 1) / R), unsigned((M + per - 1) / per));
    const size_t lds = size_t(tile) * K * 4;  // <= 64 KiB
    const auto* wb = static_cast<const uint8_t*>(w);
    if (tile == 4)
        hipLaunchKernelGGL(q5k_gemm_kernel<4>, grid, dim3(kKqThreads), lds, s, wb, x, ldx, y, resid, M, N, int(K), ldy, R, per);
    else if (tile == 2)
        hipLaunchKernelGGL(q5k_gemm_kernel<2>, grid, dim3(kKqThreads), lds, s, wb, x, ldx, y, resid, M, N, int(K), ldy, R, per);
    else
        hipLaunchKernelGGL(q5k_gemm_kernel<1>, grid, dim3(kKqThreads), lds, s, wb, x, ldx, y, resid, M, N, int(K), ldy, R, per);
}

void launch_kquant_dequant_rows(int type, const void* w, int64_t N, int64_t K, const int32_t* ids, int64_t n, float* out, hipStream_t s) {
    hipLaunchKernelGGL(kq_dequant_rows_kernel, dim3(unsigned(K / 256), unsigned(n)), dim3(256), 0, s, type, static_cast<const uint8_t*>(w), N, int(K), ids, out);
}

}  // namespace hero
