// gemm_tall.h -- a few tokens by a tall weight (a verification batch's lm_head) on
// the int8 matrix pipe, straight from the GEMV layout; included by zlm_kernels.hip.
#pragma once

typedef float v4f __attribute__((ext_vector_type(4)));

// out[t*rows + r] for 3 to 8 tokens in the int path's arithmetic (reference
// kernels/quantized.zig:49-55, :79-87, :111-123).  One 16-wave workgroup per CU
// quantizes the activations into LDS itself and its waves then walk 16-row tiles
// on their own: no barrier, no partial sums between waves, and a tile's first
// loads are in flight while the previous one computes.
//
// A step is 64 B of payload of each of the 16 rows: lane l holds 16 B (chunk l/16)
// of row l % 16, as the B operand of v_mfma_i32_16x16x64_i8.  Its K = 64 spans
// several scale blocks, so the A operand's rows are (token, block) pairs with zeros
// outside the row's own block, and the blocks' dots come out in separate rows:
//   q4_k  a chunk's low nibbles are one block's, its high another's: two products,
//         rows = 2 blocks x 8 tokens;
//   q4_0, q4_1  a chunk is a block: its low and high nibbles accumulate, rows =
//         4 blocks x 4 tokens, a second set of products from the fifth token.
// Each lane's four results belong to its own row and to its own chunk's block(s):
// the scales it loaded beside the chunk, and four tokens' dx (and dx sum q, for the
// min-carrying quants), one LDS read.
//
// The zeros are one 16-byte place that the lanes outside read; the reads of a step
// are constants apart, so that place is as long as an iteration.
//
// Bound: the payload's reads, 16 rows x 64 B an instruction (twice the cache lines
// a contiguous 1 KiB touches): q4_k 262144 x 3840 x 8 runs at 4.5 TB/s, 130 us,
// where the rate of a large copy, 5.15 TB/s, would give 113 (VALU instructions fill
// 56 us of it, the matrix pipe 6).  The small-M GEMM took 269 (its 32-token
// products and their scaling are VALU work for 24 tokens that are not there, and
// its workgroups drain at their ends); q4_0 151936 x 4096 x 8 121 -> 78, q4_1 142
// (the token GEMV) -> 82.  What mattered: each scale is loaded by one lane and
// handed on by a shuffle (each lane loading its own: 136 and 102 us for 130 and
// 80 at q4_k 262144 x 3840 and 151936 x 4096), loads without the streaming hint
// (its lines are read in two halves: 152 us with it), and tiles dealt to the CUs
// before their waves (16 tiles a workgroup first: q4_k 32768 x 4096 x 8 28 us for
// 21).  Three or four iterations in flight instead of two change nothing at
// 262144 x 3840 and cost 2 us at 32768 rows.  q8_0 gained nothing (246 -> 231, 81 ->
// 84 at 65536 x 5120) and stays with the small-M GEMM.
template <int QT>
struct Tall {
    static constexpr bool MIN = gemm_has_min(QT);
    static constexpr bool PAIRS = QT == Q4_K;       // rows = 2 blocks x 8 tokens
    static constexpr int SB = MIN ? 64 : 32;        // scale bytes of a block in LDS: 8 dx (, 8 dx sum q)
    static constexpr int NS = MIN ? 2 : 1;          // scale words a lane loads for an iteration
    static constexpr int NACC = PAIRS ? 1 : 2;
};
constexpr int kTallWaves = 16, kTallDepth = 2;  // iterations in flight
// An iteration: 128 B of a row's payload, in two steps; its activation bytes in LDS.
constexpr uint32_t kTallElems = 256, kTallIter = kTallElems * 8, kTallStep = kTallIter / 2;

// LDS offset of elements e..e+3 of token t.
template <int QT>
__device__ __forceinline__ uint32_t tall_pos(uint32_t e, uint32_t t) {
    const uint32_t it = e / kTallElems, r = e % kTallElems;
    if constexpr (QT == Q4_K) {
        const uint32_t grp = r / 64, hi = r / 32 % 2, c = 2 * (grp % 2) + r / 16 % 2;
        return it * kTallIter + grp / 2 * kTallStep + hi * 512 + c * 128 + t * 16 + r % 16;
    } else {
        const uint32_t b = r / 32, hi = r / 16 % 2;
        return it * kTallIter + b / 4 * kTallStep + (t / 4 * 2 + hi) * 256 + b % 4 * 64 + t % 4 * 16 + r % 16;
    }
}

template <int QT, int KCAP>
__device__ __forceinline__ void gemm_tall(const uint8_t* __restrict__ w, const uint8_t* __restrict__ d,
                                          const float* __restrict__ x, float* __restrict__ out, uint32_t rows,
                                          uint32_t m, uint32_t nb) {
    using T = Tall<QT>;
    __shared__ __attribute__((aligned(16))) uint8_t qa[KCAP * 8 + kTallIter];
    __shared__ __attribute__((aligned(16))) uint8_t sa[KCAP / 32 * T::SB];
    constexpr uint32_t kZero = KCAP * 8;
    const uint32_t lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
    const uint32_t wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t k = nb * 32, ni = (k + kTallElems - 1) / kTallElems;
    const uint32_t row_w = nb * 16;                                // bytes of a row's payload,
    const uint32_t row_d = QT == Q4_K ? nb / 8 * 20 : nb * (QT == Q4_1 ? 4 : 2);  // of its scales
    const uint32_t ntiles = (rows + 15) / 16, tstride = gridDim.x * kTallWaves;

    struct Frag16 {
        uint4 q[2];
        uint32_t s[T::NS];
    };
    auto load = [&](Frag16& f, uint32_t tile, uint32_t it) {
        tile = min(tile, ntiles - 1);  // past the last: its loads are not used
        const uint32_t r = min(r16, rows - 1 - tile * 16);  // rows past the last repeat it
        const uint8_t* wt = w + static_cast<size_t>(tile) * 16 * row_w;
        const uint8_t* dt = d + static_cast<size_t>(tile) * 16 * row_d;
        uint32_t c0 = it * 8 + g, c1 = c0 + 4;
        if constexpr (QT != Q4_K) {  // q4_k rows are whole iterations
            c0 = min(c0, nb - 1);
            c1 = min(c1, nb - 1);
        }
        f.q[0] = ld16<false>(wt + (r * row_w + c0 * 16));
        f.q[1] = ld16<false>(wt + (r * row_w + c1 * 16));
        // the row's scales of the iteration, a part per lane
        if constexpr (QT == Q4_K) {  // record words g, g + 1
            const uint32_t* rec = reinterpret_cast<const uint32_t*>(dt + (r * row_d + it * 20)) + g;
            f.s[0] = rec[0];
            f.s[1] = rec[1];
        } else if constexpr (QT == Q4_1) {  // blocks 2g, 2g + 1
            const uint32_t* p = reinterpret_cast<const uint32_t*>(dt + r * row_d) + min(it * 8 + 2 * g, nb - 2);
            f.s[0] = p[0];
            f.s[1] = p[1];
        } else {  // q4_0: blocks 2g, 2g + 1
            f.s[0] = *reinterpret_cast<const uint32_t*>(dt + (r * row_d + min(it * 8 + 2 * g, nb - 2) * 2));
        }
    };
    uint32_t tile = blockIdx.x + gridDim.x * wid;
    Frag16 f[kTallDepth];
    uint32_t ltile = tile, lit = 0;  // the next loads' place
    auto advance = [&] {
        if (++lit == ni) {
            lit = 0;
            ltile += tstride;
        }
    };
#pragma unroll
    for (int j = 0; j < kTallDepth; j++) {
        load(f[j], ltile, lit);
        advance();
    }

    // The activations: thread i's float4 i of every token (8 lanes a block).
    for (uint32_t i = threadIdx.x; i < ni * kTallElems / 4; i += blockDim.x) {
        float4 v[8];
        const bool in = 4 * i < k;
#pragma unroll
        for (uint32_t t = 0; t < 8; t++)
            v[t] = reinterpret_cast<const float4*>(x + static_cast<size_t>(min(t, m - 1)) * k)[in ? i : 0];
#pragma unroll
        for (uint32_t t = 0; t < 8; t++) {
            if (!(in && t < m)) v[t] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            float dx;
            int32_t s;
            const uint32_t q = q8_quant4(v[t], dx, s);
            s = sum8(s);
            *reinterpret_cast<uint32_t*>(qa + tall_pos<QT>(4 * i, t)) = q;
            if (i % 8 == 0) {
                float* o = reinterpret_cast<float*>(sa + i / 8 * T::SB);
                o[t] = dx;
                if constexpr (T::MIN) o[8 + t] = dx * static_cast<float>(s);
            }
        }
    }
    for (uint32_t i = threadIdx.x; i < kTallIter / 4; i += blockDim.x) *reinterpret_cast<uint32_t*>(qa + kZero + 4 * i) = 0;
    __syncthreads();

    // This lane's A operand: the row r16's token and block, zeros outside its block's chunks.
    const bool mine = T::PAIRS ? r16 / 8 == g / 2 : r16 / 4 == g;
    const uint32_t a0 = mine ? (T::PAIRS ? g * 128 + r16 % 8 * 16 : g * 64 + r16 % 4 * 16) : kZero;
    const uint32_t astep = mine ? kTallIter : 0;
    // The scales of its results (rows 4g..4g+3 of the product).
    const uint32_t s0 = T::PAIRS ? g / 2 * 2 * T::SB + g % 2 * 16 : g * T::SB;

    auto a_at = [&](uint32_t o) { return *reinterpret_cast<const v4i*>(qa + o); };
    auto s_at = [&](uint32_t o) { return *reinterpret_cast<const float4*>(sa + o); };
    v4f acc[kTallDepth][T::NACC];  // a chain of sums per turn
    auto clear = [&] {
#pragma unroll
        for (int s = 0; s < T::NACC * kTallDepth; s++) acc[s / T::NACC][s % T::NACC] = v4f{};
    };
    const v4i zi = {};
    auto scaled = [&](v4f t, v4i dot, float dw, float4 dx) {  // t + (dw dx) dot
        t[0] = fmaf(dw * dx.x, static_cast<float>(dot[0]), t[0]);
        t[1] = fmaf(dw * dx.y, static_cast<float>(dot[1]), t[1]);
        t[2] = fmaf(dw * dx.z, static_cast<float>(dot[2]), t[2]);
        t[3] = fmaf(dw * dx.w, static_cast<float>(dot[3]), t[3]);
        return t;
    };
    auto minned = [&](v4f t, float mn, float4 xs) {  // t + mn xs
        t[0] = fmaf(mn, xs.x, t[0]);
        t[1] = fmaf(mn, xs.y, t[1]);
        t[2] = fmaf(mn, xs.z, t[2]);
        t[3] = fmaf(mn, xs.w, t[3]);
        return t;
    };
    // An iteration's terms are summed before they meet the row's sums.
    auto compute = [&](const Frag16& f, uint32_t it, v4f (&acc)[T::NACC]) {
        const uint32_t pa = a0 + it * astep, ps = s0 + it * (kTallElems / 32 * T::SB);
        v4f t[T::NACC];
#pragma unroll
        for (int s = 0; s < T::NACC; s++) t[s] = v4f{};
        // this lane's chunks' scales (one a step), from the lanes that loaded them
        const int from[2] = {static_cast<int>(r16 + 16 * (g / 2)), static_cast<int>(r16 + 16 * (2 + g / 2))};
        uint32_t sc[2], dm = 0;
#pragma unroll
        for (int st = 0; st < 2; st++) {
            sc[st] = __shfl(f.s[T::NS - 1], from[st], kWave);
            if constexpr (QT == Q4_0) sc[st] >>= 16 * (g % 2);
            if constexpr (QT == Q4_1) {
                const uint32_t even = __shfl(f.s[0], from[st], kWave);
                sc[st] = g % 2 ? sc[st] : even;
            }
        }
        if constexpr (QT == Q4_K) dm = __shfl(f.s[0], static_cast<int>(r16), kWave);
#pragma unroll
        for (uint32_t st = 0; st < 2; st++) {
            const uint4 q = f.q[st];
            v4i lo, hi;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t v = (&q.x)[j];
                if constexpr (QT == Q4_0) {  // 16 (n - 8), undone at the store
                    lo[j] = static_cast<int>(((v << 4) & 0xF0F0F0F0u) ^ 0x80808080u);
                    hi[j] = static_cast<int>((v & 0xF0F0F0F0u) ^ 0x80808080u);
                } else {
                    lo[j] = static_cast<int>(v & 0x0F0F0F0Fu);
                    hi[j] = static_cast<int>((v >> 4) & 0x0F0F0F0Fu);
                }
            }
            if constexpr (QT == Q4_K) {
                const v4i dlo = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_at(pa + st * kTallStep), lo, zi, 0, 0, 0);
                const v4i dhi = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_at(pa + st * kTallStep + 512), hi, zi, 0, 0, 0);
                const float dw = h2f(dm), mn = -h2f(dm >> 16);
                const uint32_t sm = sc[st], p = ps + st * 4 * T::SB;
                t[0] = scaled(t[0], dlo, dw * ub(sm, 0), s_at(p));
                t[0] = scaled(t[0], dhi, dw * ub(sm, 1), s_at(p + T::SB));
                t[0] = minned(t[0], mn * ub(sm, 2), s_at(p + 32));
                t[0] = minned(t[0], mn * ub(sm, 3), s_at(p + T::SB + 32));
            } else {
                const uint32_t s = it * 8 + st * 4 + g < nb ? sc[st] : 0u;
#pragma unroll
                for (int set = 0; set < 2; set++) {
                    if (set && m <= 4) continue;
                    const uint32_t o = pa + st * kTallStep + set * 512, p = ps + st * 4 * T::SB + set * 16;
                    v4i dot = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_at(o), lo, zi, 0, 0, 0);
                    dot = __builtin_amdgcn_mfma_i32_16x16x64_i8(a_at(o + 256), hi, dot, 0, 0, 0);
                    t[set] = scaled(t[set], dot, h2f(s), s_at(p));
                    if constexpr (QT == Q4_1) t[set] = minned(t[set], h2f(s >> 16), s_at(p + 32));
                }
            }
        }
#pragma unroll
        for (int s = 0; s < T::NACC; s++) acc[s] += t[s];
    };
    auto finish = [&](uint32_t tl) {
        const uint32_t r = tl * 16 + r16;
        constexpr float kOut = QT == Q4_0 ? 0.0625f : 1.0f;
#pragma unroll
        for (int s = 0; s < T::NACC; s++) {
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                v[i] = acc[0][s][i] + acc[1][s][i];
                v[i] += __shfl_xor(v[i], 32, kWave);
                if constexpr (!T::PAIRS) v[i] += __shfl_xor(v[i], 16, kWave);
            }
            if constexpr (T::PAIRS) {  // lanes 0-31 hold tokens 4g..4g+3
#pragma unroll
                for (uint32_t i = 0; i < 4; i++)
                    if (lane < 32 && r < rows && 4 * g + i < m) out[static_cast<size_t>(4 * g + i) * rows + r] = v[i];
            } else {  // every lane all four of the set: lane group g stores token 4s + g
                const float o = g == 0 ? v[0] : g == 1 ? v[1] : g == 2 ? v[2] : v[3];
                if (r < rows && 4 * s + g < m) out[static_cast<size_t>(4 * s + g) * rows + r] = o * kOut;
            }
        }
    };
    clear();
    uint32_t it = 0;
    auto done = [&] {  // after an iteration: the tile's last stores its sums
        if (++it == ni) {
            finish(tile);
            clear();
            it = 0;
            tile += tstride;
        }
    };
    // Whole turns only: a way out in the middle would join the loop's end, and the
    // waits would count the loads of its path.  Tiles past the last store nothing.
    while (tile < ntiles) {
#pragma unroll
        for (int j = 0; j < kTallDepth; j++) {
            __builtin_amdgcn_sched_barrier(0);
            compute(f[j], it, acc[j]);
            __builtin_amdgcn_sched_barrier(0);
            load(f[j], ltile, lit);
            advance();
            done();
        }
    }
}
