// gemm_fp6.h -- the min-carrying nibble quants' (q4_1, q4_k) wide prefill GEMM on
// the fp6 matrix pipe; included by zlm_kernels.hip after the int8 GEMMs, whose
// tiled weights it shares.
//
// zlm's int path (reference kernels/quantized.zig:49-55, :79-87, :111-123 over
// the activation quantizer of matvec/layout.zig:458-476) needs, per 32-element
// block, the exact integer dot of the block's quants with the token's q8
// activations q, then one scaled add per output.  On the int8 MFMA the dot
// comes out in int32 and every output pays a convert and an fma.  Here it
// comes out in f32, exactly, and the convert is gone:
//   * fp6 e2m3 in units of 1/8 holds every integer -15..15, its code being
//     sign << 5 | magnitude (0..7 are its subnormals, 8..15 its first binade);
//   * q = 16 hi + lo with hi, lo in -8..8, and a weight quant n is 0..15: all
//     of them are fp6 values;
//   * v_mfma_scale_f32_32x32x64_f8f6f4 takes K = 64 at the rate of the int8
//     32x32x32: the lower K half carries hi times the weights, the upper half
//     lo times the same weights, and the block scales undo the units and the
//     16.  All products are integers below 2^11 and a block's sums stay below
//     2^16, so f32 holds them exactly (checked on the chip over 204,800 block
//     dots, the extremes included).
// q4_0 gains nothing from it (its int8 form carries no min term, and signed
// quants cost more to expand: 12288 x 4096 x 512 72.5 us int8, 70.4 fp6; x 1999
// 265 and 271).
//
// Activations (zlm_quantize_fp6_tiled): per 128 tokens (four tiles of 32) and
// block pair one record of whole 1 KiB runs, which a GEMM stage copies into
// LDS as it is:
//   [4 tiles][2 blocks][64 lanes][16 B]  the first 16 bytes of lane l's 24: token
//       l % 32's 32 fp6 codes (field j at bit 6j), the hi parts in lanes 0-31,
//       the lo parts in 32-63; which element sits in which field is
//       fp6_expand's order;
//   [4][2][64][8 B]  the other 8 bytes, the second block's with its halves
//       exchanged (so that no two reads of a lane are a constant apart: the
//       compiler would join them into one read and copy the halves apart);
//   [4][2][32]  dx, then [4][2][32] dx * sum q.
// Blocks past the row's end and tokens past the last are zeros.
#pragma once

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v8i __attribute__((ext_vector_type(8)));

constexpr uint32_t kFp6Tail = 8192, kFp6Dx = 12288, kFp6Xs = 13312, kFp6Record = 14336;  // offsets in a record, its size
constexpr uint32_t kFp6W = 768;  // bytes of a 32-row tile's expanded block in LDS

// E8M0 block scales of the K halves: the units of 1/8 and, for hi, the 16.
constexpr int kFp6ScaleHi = 127 + 7, kFp6ScaleLo = 127 + 3, kFp6ScaleW = 127 + 3;

__device__ __forceinline__ uint32_t fp6_code(int v) { return (v < 0 ? 32u : 0u) | static_cast<uint32_t>(v < 0 ? -v : v); }

// Two dwords of a tile's nibbles (16 elements) to 96 bits of fp6 fields.
// Nibbles sit every four bits, fields every six: of w0's nibbles 0, 3, 6 are
// in place in the first dword, 1, 4, 7 in the second and 2, 5 in the third; of
// w1's, moved up two bits (a rotate: nibble 7 straddles the first two), 1, 4,
// 7 / 2, 5 / 0, 3, 6.  The element of field j follows: with w0 holding elements
// 0-3 in its low and 16-19 in its high nibbles and w1 4-7 and 20-23,
//   fields 4q   elements 0-3 in the order 0, 3, 2, 1      (q = 0..3)
//   fields 4q+1 elements 20-23:           0, 3, 2, 1
//   fields 4q+2 elements 16-19:           1, 0, 3, 2
//   fields 4q+3 elements 4-7:             2, 1, 0, 3
// and w2, w3 likewise eight elements on.
constexpr uint32_t nibbles(uint32_t set) {  // the bits of nibbles p in `set`
    uint32_t m = 0;
    for (int p = 0; p < 8; p++)
        if ((set >> p) & 1u) m |= 0xFu << (4 * p);
    return m;
}
constexpr uint32_t rotl32(uint32_t v, int n) { return (v << n) | (v >> (32 - n)); }
constexpr uint32_t kP036 = 0x49, kP147 = 0x92, kP25 = 0x24;
__device__ __forceinline__ uint32_t rotate_left(uint32_t v, int n) { return __builtin_rotateleft32(v, n); }

__device__ __forceinline__ void fp6_expand(uint32_t w0, uint32_t w1, uint32_t& o0, uint32_t& o1, uint32_t& o2) {
    const uint32_t r = rotate_left(w1, 2);
    o0 = (w0 & nibbles(kP036)) | (r & ((nibbles(kP147) << 2)));
    o1 = (w0 & nibbles(kP147)) | (r & ((nibbles(kP25) << 2) | 3u));
    o2 = (w0 & nibbles(kP25)) | (r & (nibbles(kP036) << 2));
}

__device__ __forceinline__ v8i fp6_frag(v4i a, v2i b) { return v8i{a.x, a.y, a.z, a.w, b.x, b.y, 0, 0}; }

// A block's exact integer dots (f32) of 32 tokens by 32 rows: tokens in the
// result registers, t = 8*(i/4) + 4*(lane/32) + i%4, rows r = lane%32.
__device__ __forceinline__ v16f fp6_dot(const v8i a, const v8i w, int scale_a) {
    const v16f z = {};
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, w, z, 2, 2, 0, scale_a, 0, kFp6ScaleW);
}

// ---- the wide tiled GEMM -----------------------------------------------------
// out[t*rows + r] = sum_b dw[r,b] dx[t,b] dot[t,r,b] + mn[r,b] xs[t,b], xs = dx sum q.
//
// One workgroup per CU owns 128 tokens x 192 rows with 12 waves, three per
// SIMD; a wave owns one token tile x two row tiles.  A wave's unit of work is a
// row tile's block pair: two fp6 MFMAs, one v_mfma_f32_32x32x1_2b_f32 for both
// blocks' scale matrices dx (x) dw (lanes 0-31 give the first block's vectors,
// 32-63 the second's), 32 fmas, one K = 2 f32 product that adds the min terms, and
// 16 adds to the sums.  (Straight into the sums, the fmas and the min product took
// 347 us at 15360 x 3840 x 1999 where this form took 370, but round three times a pair at the
// sums' size: 2.8e-7 against 64 bits, where the int8 form has 2.1e-7 and this
// 1.5e-7.)
//
// Operands go through LDS: the runs a wave needs per block would take the
// CU's 64 B/clk L1 longer to deliver than the block takes to compute.  A stage
// is one block pair.  The weights' nibbles are expanded to fp6 codes on their
// way in (two lanes a row; each wave one row tile's block, shared by the four
// waves of that tile).  Three buffers: in stage s the waves read s and write
// s + 2, so one barrier a stage suffices; global loads run a stage further ahead,
// in registers (two stages ahead took 373 us where this took 370).
//
// Bound: VALU issue and the matrix pipe, one after the other.  A wave's stage has 116
// VALU instructions (96 fmas and adds, the expansion and the stores: 464 cycles) and 8
// MFMAs (384 cycles: the dots, the scale matrices and the min terms 128 each), and only
// a tenth of the MFMA cycles run beside VALU ones: over 15360 x 3840 x 1999 the two make
// up 729,000 of a SIMD's 826,000 active cycles.  The barrier keeps the three waves'
// phases in step, and f32 MFMAs take as long as the fp6 ones for a fraction of the work.
// Against the int8 form (gemm_tiles<Q4_K>), the quantizers included, in long runs of
// products: 12288 x 4096 x 512 (a workgroup on every CU) 96 -> 92 us, 15360 x 3840 x 1999
// (five rounds) 386 -> 366; a single product after a pause 99 -> 98 and 404 -> 418, the
// int8 form gaining more from the higher clocks there.
// Measured slower: the weights' stores behind the second row tile's MFMAs instead of the
// first's (3%), the activations read through L1 without LDS, four buffers and a barrier
// every second stage, eight waves with a unit's MFMAs issued under the previous unit's
// fmas (two waves a SIMD hide less than the pipelining gains).
constexpr int kFp6RowTiles = 6, kFp6Waves = 12, kFp6Units = 2;

static_assert(2 * kFp6RowTiles == kFp6Waves, "a wave expands one row tile's block");
constexpr uint32_t kFp6Copies = kFp6Record / 1024;                         // 1 KiB copies of a record
constexpr int kFp6WaveCopies = (kFp6Copies + kFp6Waves - 1) / kFp6Waves;  // per wave
constexpr uint32_t kFp6Dw = kFp6Record + kFp6RowTiles * 2 * kFp6W, kFp6Mn = kFp6Dw + kFp6RowTiles * 256,
                   kFp6Stage = kFp6Mn + kFp6RowTiles * 256;  // a stage in LDS: record, weights, scales, mins

template <int V>
struct Const {
    static constexpr int value = V;
};

__device__ __forceinline__ uint32_t gemm_ld4(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, static_cast<int>(voff), static_cast<int>(soff), 0);
}

__device__ __forceinline__ uint2 gemm_ld8(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, static_cast<int>(voff), static_cast<int>(soff), 0);
    return make_uint2(v[0], v[1]);
}

// Offsets are 32-bit: the host sends rows of more than 2^18 blocks to the other
// GEMMs (nst * 14336 and nb * 512 stay below 2^32), and rows of fewer than 43, where
// its cost model has the tiled kernels faster (the loads of stages past the end would
// cover those too).
__device__ __forceinline__ void gemm_fp6(const uint8_t* __restrict__ wq, const uint8_t* __restrict__ wsc,
                                         const uint8_t* __restrict__ qx, float* __restrict__ out, uint32_t rows,
                                         uint32_t m, uint32_t nb) {
    constexpr int JA = kFp6WaveCopies;
    constexpr uint32_t kS = kFp6Stage;
    __shared__ __attribute__((aligned(16))) uint8_t buf[3 * kS];
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
    const uint32_t half = lane >> 5, l32 = lane & 31;

    // The workgroup's output tile: workgroups are dealt to the XCDs in turn, so
    // XCD x takes consecutive tiles of an order that walks the token tiles
    // within groups of four row tiles: its concurrent workgroups share weight
    // and activation panels in its L2.
    const uint32_t gx = gridDim.x, gy = gridDim.y, total = gx * gy;
    uint32_t id = blockIdx.y * gx + blockIdx.x;
    {
        const uint32_t xcd = id % 8, q = total / 8, rem = total % 8;
        id = xcd * q + min(xcd, rem) + id / 8;
    }
    const uint32_t per = 4 * gy, grp = id / per, in = id % per, gw = min(4u, gx - 4 * grp);
    const uint32_t bx = __builtin_amdgcn_readfirstlane(4 * grp + in % gw), by = __builtin_amdgcn_readfirstlane(in / gw);
    const uint32_t rt0 = kFp6RowTiles * bx, rlast = (rows + 31) / 32 - 1;  // row tiles past the last repeat it
    const uint32_t nst = (nb + 1) / 2;  // stages

    // The operands' buffers, bounded so that weights past the row's end are
    // zeros, their scales among them (activations past it re-read the last stage).
    // LDS offsets are per-lane bases, fixed for the whole loop, plus constants (the
    // stages are unrolled over the buffers).
    // (The scalar offsets of stages past the end are held at the buffers' sizes:
    // the bounds check subtracts them from the size.)
    const __amdgpu_buffer_rsrc_t ra = gemm_rsrc(qx + static_cast<size_t>(by) * nst * kFp6Record, nst * kFp6Record);
    uint32_t ai[JA], adst[JA];  // this wave's copies (a wave with none left repeats the last)
#pragma unroll
    for (int j = 0; j < JA; j++) {
        ai[j] = min(static_cast<uint32_t>(j * kFp6Waves) + wid, kFp6Copies - 1u) * 1024;
        adst[j] = ai[j] + lane * 16;
    }
    // The row tile's block this wave expands (the waves with fewer copies first),
    // its scales with it; two lanes a row: elements 0-7 and 16-23, the others.
    // Even lanes produce the row's dwords 0-2 (of the first 16 bytes), odd lanes 3
    // and the tail's two.
    const uint32_t h = lane & 1, row = lane >> 1;
    const uint32_t wblk = (kFp6Waves - 1 - wid) % 2, wtile = (kFp6Waves - 1 - wid) / 2;
    const size_t first =
        static_cast<size_t>(__builtin_amdgcn_readfirstlane(min(rt0 + wtile, rlast))) * nb + min(wblk, nb - 1);
    const uint32_t left = __builtin_amdgcn_readfirstlane(nb - wblk);  // the row's blocks from there on (nb >= 1)
    const __amdgpu_buffer_rsrc_t rw = gemm_rsrc(wq + first * 512, left * 512);
    const __amdgpu_buffer_rsrc_t rs = gemm_rsrc(wsc + first * 256, left * 256);
    const uint32_t wmain = kFp6Record + wtile * 2 * kFp6W + wblk * 512 + row * 16;
    const uint32_t wtail = kFp6Record + wtile * 2 * kFp6W + 1024 + wblk * 256 + (row ^ (16 * wblk)) * 8;
    const uint32_t wd0 = h ? wmain + 12 : wmain, wd1 = h ? wtail : wmain + 4, wd2 = h ? wtail + 4 : wmain + 8;
    const uint32_t wds = (h ? kFp6Mn : kFp6Dw) + wtile * 256 + wblk * 128 + row * 4;

    struct Staged {
        uint4 a[JA];
        uint2 w;
        uint32_t d;  // the row's scale (f32 bits), in its odd lane the min
    };
    Staged st;
    auto load = [&](Staged& v, uint32_t s) {
        const uint32_t sa = min(s, nst - 1) * kFp6Record, bw = min(2 * s, left);
#pragma unroll
        for (int j = 0; j < JA; j++) v.a[j] = gemm_ld16(ra, lane * 16, sa + ai[j]);
        v.w = gemm_ld8(rw, lane * 8, bw * 512);
        v.d = gemm_ld4(rs, lane * 4, bw * 256);
    };
    auto store = [&](const Staged& v, uint32_t o) {
#pragma unroll
        for (int j = 0; j < JA; j++) *reinterpret_cast<uint4*>(buf + adst[j] + o) = v.a[j];
        uint32_t e0, e1, e2;
        fp6_expand(v.w.x, v.w.y, e0, e1, e2);
        *reinterpret_cast<uint32_t*>(buf + wd0 + o) = e0;
        *reinterpret_cast<uint32_t*>(buf + wd1 + o) = e1;
        *reinterpret_cast<uint32_t*>(buf + wd2 + o) = e2;
        *reinterpret_cast<uint32_t*>(buf + wds + o) = v.d;
    };

    const uint32_t wt = wid % 4, wr = wid / 4 * kFp6Units;  // this wave's token tile and first row tile
    const int scale_a = half ? kFp6ScaleLo : kFp6ScaleHi;
    const uint8_t *pa = buf + wt * 2048 + lane * 16, *pt0 = buf + kFp6Tail + wt * 1024 + lane * 8,
                  *pt1 = buf + kFp6Tail + wt * 1024 + 512 + (lane ^ 32) * 8, *px = buf + kFp6Dx + wt * 256 + lane * 4;
    const uint8_t* pw = buf + kFp6Record + wr * 2 * kFp6W;
    const uint8_t *pw0 = pw + l32 * 16, *pwt0 = pw + 1024 + l32 * 8, *pwt1 = pw + 1280 + (l32 ^ 16) * 8,
                  *pd = buf + kFp6Dw + wr * 256 + lane * 4;
    v16f acc[kFp6Units];
#pragma unroll
    for (int u = 0; u < kFp6Units; u++) acc[u] = v16f{};
    const v32f zf = {};

    load(st, 0);
    store(st, 0);
    load(st, 1);
    store(st, kS);
    load(st, 2);
    sk_barrier();
    // One stage (K of three in turn).
    auto stage = [&](auto turn, uint32_t s) {
        constexpr int K = decltype(turn)::value;
        constexpr uint32_t cur = K * kS, wrt = (K + 2) % 3 * kS;
        const v8i a0 = fp6_frag(*reinterpret_cast<const v4i*>(pa + cur), *reinterpret_cast<const v2i*>(pt0 + cur));
        const v8i a1 = fp6_frag(*reinterpret_cast<const v4i*>(pa + cur + 1024), *reinterpret_cast<const v2i*>(pt1 + cur));
        const float x = *reinterpret_cast<const float*>(px + cur);
        const float xs = *reinterpret_cast<const float*>(px + cur + (kFp6Xs - kFp6Dx));
#pragma unroll
        for (int u = 0; u < kFp6Units; u++) {
            const uint32_t ou = cur + u * 2 * kFp6W;
            const v8i w0 = fp6_frag(*reinterpret_cast<const v4i*>(pw0 + ou), *reinterpret_cast<const v2i*>(pwt0 + ou));
            const v8i w1 = fp6_frag(*reinterpret_cast<const v4i*>(pw0 + ou + 512), *reinterpret_cast<const v2i*>(pwt1 + ou));
            const float dw = *reinterpret_cast<const float*>(pd + cur + u * 256);
            const v32f c = __builtin_amdgcn_mfma_f32_32x32x1f32(x, dw, zf, 0, 0, 0);
            const v16f f0 = fp6_dot(a0, w0, scale_a), f1 = fp6_dot(a1, w1, scale_a);
            const float mn = *reinterpret_cast<const float*>(pd + cur + u * 256 + (kFp6Mn - kFp6Dw));
            v16f t;
#pragma unroll
            for (int i = 0; i < 16; i++) t[i] = fmaf(c[16 + i], f1[i], c[i] * f0[i]);
            t = __builtin_amdgcn_mfma_f32_32x32x2f32(xs, mn, t, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 16; i++) acc[u][i] += t[i];
            asm volatile("" : "+v"(acc[u]));  // keep the sums one register tuple
            if (u == 0) {
                store(st, wrt);
                load(st, s + 3);
            }
        }
        sk_barrier();
    };
    for (uint32_t s = 0;; s += 3) {
        stage(Const<0>{}, s);
        if (s + 1 >= nst) break;
        stage(Const<1>{}, s + 1);
        if (s + 2 >= nst) break;
        stage(Const<2>{}, s + 2);
        if (s + 3 >= nst) break;
    }
#pragma unroll
    for (int u = 0; u < kFp6Units; u++) {
        const uint32_t r = 32 * (rt0 + wr + u) + l32;
        if (r < rows) {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const uint32_t t = 128 * by + 32 * wt + 8 * (i / 4) + 4 * half + (i % 4);
                if (t < m) out[static_cast<size_t>(t) * rows + r] = acc[u][i];
            }
        }
    }
}
