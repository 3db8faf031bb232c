// Q8_0 products of fewer than 32 positions (17 to 31 of matrices of many rows share lng_q8_mid's tiles): lng_q8_norm_frag,
// lng_q8_few*, lng_q8_one*, lng_q8_tall*. (Included by lng_kernels.hip after lng_q8_mid.h; see there for how a product goes through the matrix unit.)

// x[n][x_stride] f32 as the A operands of lng_q8_few and lng_q8_mid, RMS-normalised on the way if norm_w is set
// (x / sqrt(mean(x^2) + eps) * w): one workgroup per position, lng_q8_frag_x's layout. Rows that pad n to whole groups
// are not written: what the scratch holds there goes into rows of the products that are not stored.
extern "C" __global__ __launch_bounds__(512) void lng_q8_norm_frag(lng_k_q8_split a) {
    __shared__ float s_norm[8];
    const uint32_t p = blockIdx.x, blocks = a.cols / 32u, chunks = a.cols / 8u;
    const float *xp = a.x + (uint64_t)p * a.x_stride;
    float x[8] = {};
    const uint32_t first = threadIdx.x;
    auto load = [&](uint32_t chunk) {
        const float4 u = *(const float4 *)(xp + 8u * chunk), v = *(const float4 *)(xp + 8u * chunk + 4u);
        x[0] = u.x, x[1] = u.y, x[2] = u.z, x[3] = u.w, x[4] = v.x, x[5] = v.y, x[6] = v.z, x[7] = v.w;
    };
    float scale = 0.0f;
    if (a.norm_w) { // uniform
        float ss = 0.0f;
        for (uint32_t c = first + 512u; c < chunks; c += 512u) {
            load(c);
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
        }
        if (first < chunks) {
            load(first);
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
        if ((threadIdx.x & 63u) == 0) s_norm[threadIdx.x >> 6] = ss;
        __syncthreads();
        float total = 0.0f;
#pragma unroll
        for (int w = 0; w < 8; ++w) total += s_norm[w];
        scale = 1.0f / sqrtf(total / (float)a.cols + a.eps);
    } else if (first < chunks) {
        load(first);
    }
    for (uint32_t c = first; c < chunks; c += 512u) {
        if (c != first) load(c);
        if (a.norm_w) {
            const float4 u = *(const float4 *)(a.norm_w + 8u * c), v = *(const float4 *)(a.norm_w + 8u * c + 4u);
            const float w[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = x[e] * scale * w[e];
        }
        bf16x8 hi, lo;
        q8_split8(x, hi, lo);
        const uint32_t lane = 16u * q8_mid_chunk(c & 3u) + (p & 15u); // (q8_mid_chunk is its own inverse)
        uint4 *to = (uint4 *)a.hi + ((uint64_t)(p >> 4) * blocks + (c >> 2)) * 128u + lane;
        to[0] = __builtin_bit_cast(uint4, hi);
        to[64] = __builtin_bit_cast(uint4, lo);
    }
}

// The matrix, in the workgroup's run of 16 rows: wavefront w of NW takes a contiguous run of block pairs; a lane loads 16
// bytes of a row at once, which one swap of register halves makes the B operands of both blocks (lng_q8_mid).
// The rows' scales wait in LDS, both of a pair in one word, rows an odd number of words apart (no two of the sixteen in
// one bank); rows of more than 512 blocks read theirs from memory.
#define Q8F_SC_BLOCKS 512u
__device__ __forceinline__ uint32_t q8_few_sc_words(uint32_t blocks) { return ((blocks + 1u) / 2u) | 1u; }

// HEADS: the tile's sixteen rows are 8 q .. 8 q + 7 and 32 + 8 q .. of a head of 64 (tile = 4 head + q): what rotation by
// halves pairs is in one tile.
template <bool HEADS> __device__ __forceinline__ uint32_t q8_tile_row(uint32_t tile) { return HEADS ? (tile >> 2) * 64u + (tile & 3u) * 8u : tile * 16u; }
template <bool HEADS> __device__ __forceinline__ uint32_t q8_row_in(uint32_t j) { return HEADS ? (j & 7u) + (j >> 3) * 32u : j; }

template <int NW, bool HEADS = false> struct Q8Few {
    static constexpr int U = 8; // block pairs in flight: 4,096 columns in one turn of eight wavefronts
    const int8_t *w_src;
    const uint16_t *sc_rows;   // the tile's first row of scales
    uint32_t *s_sc;
    uint32_t blocks, pairs, from, to, lane, wave, j, kg, rows_here, words;
    bool staged, words_aligned;
    uint32_t sc_now[16 / NW], sc_then[16 / NW];
    uint4 w[U];

    __device__ __forceinline__ Q8Few(const lng_k_q8 &a, uint32_t tile, uint32_t *lds) : s_sc(lds) {
        lane = threadIdx.x & 63u;
        wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        j = lane & 15u;
        kg = lane >> 4;
        blocks = a.cols / 32u;
        pairs = (blocks + 1u) / 2u;
        from = wave * pairs / NW;
        to = (wave + 1u) * pairs / NW;
        const uint32_t r0 = q8_tile_row<HEADS>(tile);
        rows_here = HEADS || a.rows - r0 >= 16u ? 16u : a.rows - r0;
        const uint32_t row = q8_row_in<HEADS>(j < rows_here ? j : rows_here - 1u);
        w_src = a.codes + (uint64_t)(r0 + row) * a.cols + 16u * kg;
        sc_rows = a.scales + (uint64_t)r0 * blocks;
        staged = blocks <= Q8F_SC_BLOCKS;
        words_aligned = ((blocks & 1u) | ((uintptr_t)sc_rows & 3u)) == 0;
        words = q8_few_sc_words(blocks);
    }
    // Scales 2 word and 2 word + 1 of a row: one load, or (off a 4-byte boundary) two, which are put together where they are
    // used: nothing waits here for what it asks for.
    __device__ __forceinline__ void ask_sc(uint32_t row, uint32_t word, uint32_t &first, uint32_t &second) const {
        const uint16_t *src = sc_rows + row * blocks + 2u * word;
        if (words_aligned) { // uniform
            first = *(const uint32_t *)src;
        } else {
            first = src[0];
            if (2u * word + 1u < blocks) second = src[1];
        }
    }
    __device__ __forceinline__ uint32_t both_sc(uint32_t word, uint32_t first, uint32_t second) const { // zero past the last block
        // (low halves of both; a shift of the second alone would be moved to its load, and wait there)
        return words_aligned || 2u * word + 1u >= blocks ? first : __builtin_amdgcn_perm(second, first, 0x05040100u);
    }
    __device__ __forceinline__ uint32_t load_sc(uint32_t row, uint32_t word) const {
        uint32_t first, second;
        ask_sc(row, word, first, second);
        return both_sc(word, first, second);
    }
    __device__ __forceinline__ uint32_t sc_row(int i) const {
        const uint32_t row = wave * (16 / NW) + i;
        return q8_row_in<HEADS>(row < rows_here ? row : rows_here - 1u);
    }
    __device__ __forceinline__ void ask_scales() { // the first 64 words of the wavefront's rows, into registers
        if (!staged) return;
#pragma unroll
        for (int i = 0; i < 16 / NW; ++i) {
            if (lane < pairs) ask_sc(sc_row(i), lane, sc_now[i], sc_then[i]);
        }
    }
    __device__ __forceinline__ void stage_scales() { // and all of them to LDS
        if (!staged) return;
#pragma unroll
        for (int i = 0; i < 16 / NW; ++i) {
            uint32_t *to_row = s_sc + (wave * (16 / NW) + i) * words;
            if (lane < pairs) to_row[lane] = both_sc(lane, sc_now[i], sc_then[i]);
            for (uint32_t at = lane + 64u; at < pairs; at += 64u) to_row[at] = load_sc(sc_row(i), at);
        }
    }
    // (Nothing is put in place of what is not loaded - the products skip it too - and the first load is asked for in any case:
    // a value merged with another after a branch is copied, and the copy waits for the load.)
    __device__ __forceinline__ void ask_codes(uint32_t base) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t pair = u || base < to ? base + u : pairs - 1u;
            if (u == 0 || pair < to) { // uniform; a last pair of one block: its upper lanes load the block again
                const int64_t col = (int64_t)(64ull * pair) - (2u * pair + 1u == blocks && kg >= 2u ? 32 : 0);
                w[u] = *(const uint4 *)(w_src + col);
            }
        }
    }
    // the B operands and the scales of both blocks of a pair
    __device__ __forceinline__ void operands(int u, uint32_t pair, bf16x8 (&b)[2], float (&sc)[2]) const {
        const auto s0 = __builtin_amdgcn_permlane32_swap(w[u].x, w[u].z, false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(w[u].y, w[u].w, false, false);
        b[0] = q8_codes_to_bf16_perm(make_uint2(s0[0], s1[0]));
        b[1] = q8_codes_to_bf16_perm(make_uint2(s0[1], s1[1]));
        const uint32_t both = staged ? s_sc[j * words + pair] : load_sc(q8_row_in<HEADS>(j < rows_here ? j : rows_here - 1u), pair);
        sc[0] = f16_bits_to_f32((uint16_t)both);
        sc[1] = f16_bits_to_f32((uint16_t)(both >> 16)); // zero past an odd number of blocks
    }
};

// lng_prepare's step for one output of the q, k or v projection (which = 0, 1, 2; heads of 64, all of it rotated): bias,
// rotation with the value 32 rows away, narrowing, to the prepared queries or the cache. What it needs besides the two values
// is asked for before the product.
struct Q8Prepared {
    float bias, bias_there, c, s;
    char *to;
    // (Loads of what is absent read `any` instead: a load behind a branch would be waited for before the branch ends.)
    // ONE position is the one item, whose `start` is the row of the caches already (q8's fuse_prepare).
    template <bool ONE> static __device__ __forceinline__ lng_prepare_item item_of(const lng_k_prepare &p, uint32_t position, uint32_t &r) {
        r = ONE || p.items ? 0u : position; // a table's items are of one position each
        if constexpr (ONE) return p.first;
        else return p.items ? p.items[position] : p.first;
    }
    __device__ __forceinline__ void ask_of(const lng_k_prepare &p, uint32_t which, const lng_prepare_item &it, uint32_t r, uint32_t row, const float *any) {
        const float *b = which == 0 ? p.q_bias : which == 1 ? p.k_bias : p.v_bias;
        bias = *(b ? b + row : any);
        bias_there = *(b && which < 2u ? b + (row ^ 32u) : any);
        const float2 t = *(const float2 *)(which < 2u ? p.table + it.table_offset + ((uint64_t)r * 32u + (row & 31u)) * 8u : (const char *)any);
        c = t.x, s = t.y;
    }
    // ROW: it.start is the row of the caches already.
    template <bool ROW = false> __device__ __forceinline__ void place_of(const lng_k_prepare &p, uint32_t which, const lng_prepare_item &it, uint32_t r, uint32_t row) {
        const uint32_t es = p.out_dtype == LNG_BF16 ? 2u : 4u;
        if (which == 0) {
            to = p.q_out + it.q_out_offset + ((uint64_t)r * p.heads * 64u + row) * es;
        } else {
            const uint64_t at = ((ROW ? it.start : (it.start + r) % it.slots) * p.kv_heads * 64u + row) * es;
            to = which == 1 ? p.k_cache + it.k_cache_offset + at : p.v_cache + it.v_cache_offset + at;
        }
    }
    template <bool ONE> __device__ __forceinline__ void ask(const lng_k_prepare &p, uint32_t which, uint32_t position, uint32_t row, const float *any) {
        uint32_t r;
        const lng_prepare_item it = item_of<ONE>(p, position, r);
        ask_of(p, which, it, r, row, any);
    }
    template <bool ONE> __device__ __forceinline__ void place(const lng_k_prepare &p, uint32_t which, uint32_t position, uint32_t row) {
        uint32_t r;
        const lng_prepare_item it = item_of<ONE>(p, position, r);
        place_of<ONE>(p, which, it, r, row);
    }
    __device__ __forceinline__ void store(const lng_k_prepare &p, uint32_t which, uint32_t row, float here, float there) const {
#pragma clang fp contract(off)
        const float *b = which == 0 ? p.q_bias : which == 1 ? p.k_bias : p.v_bias;
        float x = here, y = there;
        if (b) {
            x = x + bias;
            y = y + bias_there;
        }
        if (which < 2u) x = (row & 32u) ? x * c + y * s : x * c - y * s;
        if (p.out_dtype == LNG_BF16) *(uint16_t *)to = f32_to_bf16_bits(x);
        else *(float *)to = x;
    }
};

// Bound by latencies - a start, one round trip to memory, the partial sums' way through LDS - before the reading of the
// matrix: 5,120 x 2,880 (q, k and v, 15.7 MB) with the norm, in a batch of 16 such: 2 to 16 positions 12 us with the planes' dispatch (20-27
// when each workgroup normalised and split all positions itself), 31: 14 us (38); 2,880 x 4,096 with bias and residual from
// bf16 16, 31 positions: 8.1, 10 us (13, 23), from f32 11, 16 (19, 35). One position: see q8_one_body.
// Eight wavefronts to 16 rows: two workgroups fit a compute unit, so up to 512 tiles are all in flight at once.

// 2 to 16 positions (more: 16 per blockIdx.y). Every load of a turn is asked for before its first product, the matrix's
// first: a product is one round trip to memory, not one per block.
#define Q8F_PLANES 0 // x as lng_q8_norm_frag left it
#define Q8F_BF16 1   // bf16 positions, turned into operand order through LDS that only this wavefront uses (lng_q8_mid)
#define Q8F_F32 2    // f32 positions, split (and normalised, if a.norm_w is set) by every workgroup for itself: see q8_few_direct
template <int X, int NW, bool PREPARE = false>
__device__ __forceinline__ void q8_few_body(const lng_k_q8 &a, uint32_t tile, char *s_mem, const lng_k_prepare *prepare = nullptr, uint32_t which = 0) {
    constexpr int PLANES = X == Q8F_BF16 ? 1 : 2;
    constexpr int U = Q8Few<NW>::U, D = PLANES == 2 ? (X == Q8F_F32 && PREPARE ? 2 : 3) : 6; // pairs of x in flight (what the registers hold)
    constexpr uint32_t STRIDE = 80;
    __shared__ float s_red[NW][4][64];
    __shared__ float s_norm[X == Q8F_F32 ? 16 : 1];
    Q8Few<NW, PREPARE> m(a, tile, (uint32_t *)(s_mem + (PLANES == 1 ? NW * 2u * 16u * STRIDE : 0u)));
    const uint32_t lane = m.lane, j = m.j, kg = m.kg, p0 = blockIdx.y * 16u, r0 = q8_tile_row<PREPARE>(tile);
    char *s_x = s_mem + m.wave * 2u * 16u * STRIDE;
    const uint32_t put = (lane >> 2) * STRIDE + 16u * (lane & 3u), get = j * STRIDE + 16u * q8_mid_chunk(kg);
    const uint4 *x_frag = (const uint4 *)a.x_hi + (uint64_t)blockIdx.y * m.blocks * 128u + lane;
    const uint32_t at_p = p0 + (lane >> 2) < a.n ? p0 + (lane >> 2) : a.n - 1u;
    const uint16_t *x_row = a.x_hi + (uint64_t)at_p * a.plane_stride + 8u * (lane & 3u);
    const float *x_f32 = a.x + (uint64_t)(p0 + j < a.n ? p0 + j : a.n - 1u) * a.x_stride + 8u * q8_mid_chunk(kg);
    uint4 x[D][2][PLANES]; // (Q8F_F32: eight floats until they are split)
    auto ask_x = [&](uint32_t pair, uint4 (&to)[2][PLANES]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t b = 2u * pair + h < m.blocks ? 2u * pair + h : 2u * pair;
            if constexpr (X == Q8F_BF16) {
                to[h][0] = *(const uint4 *)(x_row + 32u * b);
            } else if constexpr (X == Q8F_F32) {
                to[h][0] = *(const uint4 *)(x_f32 + 32ull * b);
                to[h][1] = *(const uint4 *)(x_f32 + 32ull * b + 4u);
            } else {
                to[h][0] = x_frag[(uint64_t)b * 128u];
                to[h][1] = x_frag[(uint64_t)b * 128u + 64u];
            }
        }
    };
    // this thread's output, and what is added to it
    const uint32_t out_p = p0 + 4u * kg + m.wave, out_row = r0 + q8_row_in<PREPARE>(j); // wavefronts 0-3: accumulator register = wavefront
    const bool mine = m.wave < 4u && out_p < a.n && j < m.rows_here;
    float *yp = a.y + (uint64_t)out_p * a.y_stride + out_row;
    float bias = 0.0f, held = 0.0f;
    if (mine && a.bias) bias = a.bias[out_row];
    if (mine && a.accumulate) held = *yp;
    float *to = a.residual + (uint64_t)out_p * a.rows + out_row; // (never with accumulate)
    if (mine && a.residual) held = *to;
    Q8Prepared ready;
    if constexpr (PREPARE) {
        if (mine) {
            ready.ask<false>(*prepare, which, out_p, out_row, (const float *)a.codes);
            ready.place<false>(*prepare, which, out_p, out_row);
        }
    }

    floatx4 y = {0.0f, 0.0f, 0.0f, 0.0f};
    const floatx4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    auto ask = [&](uint32_t base) {
        m.ask_codes(base);
#pragma unroll
        for (int u = 0; u < D; ++u) {
            if (base + u < m.to) ask_x(base + u, x[u]);
        }
    };
    m.ask_scales();
    __builtin_amdgcn_sched_barrier(0);
    ask(m.from);
    __builtin_amdgcn_sched_barrier(0);
    m.stage_scales();
    float *s_nw = (float *)(s_mem + (m.staged ? 64u * m.words : 0u));
    const bool normed = X == Q8F_F32 && a.norm_w != nullptr; // uniform
    if constexpr (X == Q8F_F32) {
        if (normed) {
            for (uint32_t c = 4u * threadIdx.x; c < a.cols; c += 4u * 64u * NW) *(float4 *)(s_nw + c) = *(const float4 *)(a.norm_w + c);
            static_assert(NW == 8, "a wavefront takes positions w and w + 8 of the sixteen");
            if (p0 + m.wave < a.n) { // uniform
                const float *x0 = a.x + (uint64_t)(p0 + m.wave) * a.x_stride;
                const bool two = p0 + m.wave + 8u < a.n; // (else the first position again)
                const float *x1 = two ? x0 + 8ull * a.x_stride : x0;
                float s0 = 0.0f, s1 = 0.0f;
#pragma unroll 2
                for (uint32_t c = 4u * lane; c < a.cols; c += 256u) {
                    const float4 v = *(const float4 *)(x0 + c), w = *(const float4 *)(x1 + c);
                    s0 += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
                    s1 += w.x * w.x + w.y * w.y + w.z * w.z + w.w * w.w;
                }
#pragma unroll
                for (int off = 32; off > 0; off >>= 1) {
                    s0 += __shfl_xor(s0, off, 64);
                    s1 += __shfl_xor(s1, off, 64);
                }
                if (lane == 0) {
                    s_norm[m.wave] = 1.0f / sqrtf(s0 / (float)a.cols + a.eps);
                    if (two) s_norm[m.wave + 8u] = 1.0f / sqrtf(s1 / (float)a.cols + a.eps);
                }
            }
        }
    }
    __syncthreads();
    const float scale = normed ? s_norm[p0 + j < a.n ? j : a.n - 1u - p0] : 1.0f;
    for (uint32_t base = m.from; base < m.to; base += U) {
        if (base != m.from) ask(base);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (base + u < m.to) {
                bf16x8 b[2];
                float sc[2];
                m.operands(u, base + u, b, sc);
                if constexpr (PLANES == 1) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) *(uint4 *)(s_x + h * 16 * STRIDE + put) = x[u % D][h][0];
#pragma unroll
                    for (int h = 0; h < 2; ++h) x[u % D][h][0] = *(const uint4 *)(s_x + h * 16 * STRIDE + get);
                }
                if constexpr (X == Q8F_F32) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const uint4 u0 = x[u % D][h][0], u1 = x[u % D][h][1];
                        float v[8] = {__uint_as_float(u0.x), __uint_as_float(u0.y), __uint_as_float(u0.z), __uint_as_float(u0.w),
                                      __uint_as_float(u1.x), __uint_as_float(u1.y), __uint_as_float(u1.z), __uint_as_float(u1.w)};
                        if (normed) {
                            const float *w = s_nw + 32u * (2u * (base + u) + h < m.blocks ? 2u * (base + u) + h : 2u * (base + u)) + 8u * q8_mid_chunk(kg);
#pragma unroll
                            for (int e = 0; e < 8; ++e) v[e] = v[e] * scale * w[e];
                        }
                        bf16x8 hi, lo;
                        q8_split8(v, hi, lo);
                        x[u % D][h][0] = __builtin_bit_cast(uint4, hi);
                        x[u % D][h][1] = __builtin_bit_cast(uint4, lo);
                    }
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    floatx4 acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(x[u % D][h][0]), b[h], zero4, 0, 0, 0);
                    if constexpr (PLANES == 2) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(x[u % D][h][1]), b[h], acc, 0, 0, 0);
                    if (h == 0 || 2u * (base + u) + 1u < m.blocks) { // uniform
#pragma unroll
                        for (int i = 0; i < 4; ++i) y[i] = __builtin_fmaf(sc[h], acc[i], y[i]);
                    }
                }
                if constexpr (D < U) {
                    if (u + D < U && base + u + D < m.to) ask_x(base + u + D, x[u % D]);
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) s_red[m.wave][i][lane] = y[i];
    __syncthreads();
    if (!mine) return;
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) sum += s_red[w][m.wave][lane];
    if (a.bias) sum = sum + bias;
    if (a.accumulate) sum = held + sum; // h + ((W x) + bias), each sum rounded as the separate dispatches round it
    *yp = sum;
    if (a.residual) *to = held + sum;
    if constexpr (PREPARE) ready.store(*prepare, which, out_row, sum, __shfl_xor(sum, 8, 64)); // (all rows of a position are mine or none)
}

// One position, on the integer matrix unit, which takes the codes as they are: widening them for the other one was most of
// the vector unit's work here. x goes in as whole numbers too: of each block of 32 columns the largest |x| sets a power of
// two, every x of the block becomes a 30-bit number of that unit (exact where it is within 2^-6 of the largest, else rounded
// at 2^-30 of it), and its four signed bytes lie in four planes in LDS. One matrix instruction multiplies 16 rows by 64 columns, two blocks: rows 0-3 of the other operand are
// the first block's planes (zero in the second's columns), rows 4-7 the second's; the next pair's go into rows 8-15 and the
// same accumulators. So lane group kg ends with the four planes' exact sums of block kg of four, and puts them together.
// The other products hold 2^-18 of each x, however small (two bf16 values; from bf16 all of it). The planes hold that much of x from
// 2^-12 of the block's largest on (bf16: 2^-22). One block in eighty of normally distributed f32 has a smaller one: what rounding
// left of such a block, as whole numbers of 2^-15 of its unit, lies in two planes more, enough for x down to 2^-26; what is still
// missing, in blocks of any spread, q8_one_rest adds. Looking for such blocks and, in most calls, adding some costs 0.3 us (without:
// 5,120 x 2,880 5.5, with: 5.8; 2,880 x 4,096 5.3 and 5.6; from bf16, where they are rare, 5.2 and 5.3).
// An x that is not finite goes through q8_one_rest as well: an infinity of f32 gives NaN (its lower bf16 value is one), of bf16
// infinities, and NaN where the code is 0, as in the other products.
// Bound by memory and by what lies before and after it: 1 us until all loads are on their way, a round trip, the matrix at the
// rate of the whole device (15.7 MB: 2.6 us), 0.8 us of sums and their way through LDS, a dispatch's start and end. In a token
// through 24 blocks (kernel trace; as two bf16 planes on the other unit / so / with the planes of the rest): 5,120 x 2,880 with norm
// and preparation 9.1 us / 7.6 / 8.2, 2,880 x 4,096 with bias and residual from bf16 7.2 / 5.5 / 5.9, from f32 7.3 / 5.2 / 6.1. Of the
// gain the whole numbers 9.1 -> 7.8 and 7.2 -> 5.9 (the sums of 4,096 columns took a wavefront 1.55 us, now 0.5), tiles of 10 to 14
// rows and x before the codes the rest.
#define Q8WHOLE_REST 15
struct Q8Whole { // eight columns, a quarter of a block; the other three are in the neighbouring lanes
    uint2 plane[4];
    float unit;    // 2^-shift; negative: the block has an x of which the planes hold less than BITS
    int32_t shift;
    bool not_finite;
    uint32_t top, low; // the block's largest, and its smallest but zero, less one
    static __device__ __forceinline__ float whole(float v, int32_t shift) { return __builtin_amdgcn_ldexpf(v, shift); }
    // what rounding leaves, in units of 2^-Q8WHOLE_REST (exact: it has no more digits than x)
    static __device__ __forceinline__ float rest(float v, int32_t shift) {
        const float w = whole(v, shift);
        return (w - __builtin_rintf(w)) * (float)(1 << Q8WHOLE_REST);
    }
    __device__ __forceinline__ bool below(uint32_t exponent) const { // whether an x is not zero and below 2^-exponent of the largest's power of two
        const uint32_t of_top = top >> 23; // (all of them below 2^-127 + exponent: what is not held is nothing in f32)
        return of_top > exponent && low < ((of_top - exponent) << 23) - 1u;
    }
    __device__ __forceinline__ void measure(const float (&x)[8]) {
        top = 0, low = ~0u;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t magnitude = __float_as_uint(x[e]) & 0x7fffffffu;
            top = top > magnitude ? top : magnitude;
            low = low < magnitude - 1u ? low : magnitude - 1u;
        }
        const uint32_t one = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0xB1, 0xf, 0xf, true); // quad_perm [1,0,3,2]
        top = top > one ? top : one;
        const uint32_t two = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)top, 0x4E, 0xf, 0xf, true); // quad_perm [2,3,0,1]
        top = top > two ? top : two;
        const uint32_t low_one = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)low, 0xB1, 0xf, 0xf, true);
        low = low < low_one ? low : low_one;
        const uint32_t low_two = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)low, 0x4E, 0xf, 0xf, true);
        low = low < low_two ? low : low_two;
    }
    // An x that is not finite is left to q8_one_rest: it becomes zero here.
    template <int BITS> __device__ __forceinline__ void make(float (&x)[8]) {
        measure(x);
        not_finite = top >= 0x7f800000u; // of the whole quad
        if (not_finite) {
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = (__float_as_uint(x[e]) & 0x7fffffffu) >= 0x7f800000u ? 0.0f : x[e];
            measure(x);
        }
        const int32_t exponent = (int32_t)(top >> 23) > 7 ? (int32_t)(top >> 23) - 127 : -120; // the unit of smaller blocks: 2^-149
        shift = 29 - exponent;
        unit = __builtin_amdgcn_ldexpf(not_finite || below(30 - BITS) ? -1.0f : 1.0f, -shift);
        uint32_t q[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) q[e] = ((uint32_t)(int32_t)__builtin_rintf(whole(x[e], shift)) + 0x00808080u) ^ 0x00808080u; // signed bytes
        uint32_t word[4][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t a = __builtin_amdgcn_perm(q[4 * h + 1], q[4 * h], 0x05010400u), b = __builtin_amdgcn_perm(q[4 * h + 1], q[4 * h], 0x07030602u);
            const uint32_t c = __builtin_amdgcn_perm(q[4 * h + 3], q[4 * h + 2], 0x05010400u), d = __builtin_amdgcn_perm(q[4 * h + 3], q[4 * h + 2], 0x07030602u);
            word[0][h] = __builtin_amdgcn_perm(c, a, 0x05040100u);
            word[1][h] = __builtin_amdgcn_perm(c, a, 0x07060302u);
            word[2][h] = __builtin_amdgcn_perm(d, b, 0x05040100u);
            word[3][h] = __builtin_amdgcn_perm(d, b, 0x07060302u);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) plane[k] = make_uint2(word[k][0], word[k][1]);
    }
    // the rest's two planes: at most 2^14 of its units, cut off
    __device__ __forceinline__ void make_rest(const float (&x)[8], uint2 (&to)[2]) const {
        uint32_t q[8], word[2][2];
#pragma unroll
        for (int e = 0; e < 8; ++e) q[e] = ((uint32_t)(int32_t)rest(x[e], shift) + 0x80u) ^ 0x80u;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t a = __builtin_amdgcn_perm(q[4 * h + 1], q[4 * h], 0x05010400u), c = __builtin_amdgcn_perm(q[4 * h + 3], q[4 * h + 2], 0x05010400u);
            word[0][h] = __builtin_amdgcn_perm(c, a, 0x05040100u);
            word[1][h] = __builtin_amdgcn_perm(c, a, 0x07060302u);
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) to[k] = make_uint2(word[k][0], word[k][1]);
    }
};

// What a block's planes and (f32) those of its rest do not hold, as two bf16 values of each x (one, exactly, where the positions are
// bf16), times the row's codes and scale; every lane group returns the same. x is read and normalised once more.
template <bool BF16>
__device__ __forceinline__ float q8_one_rest(const lng_k_q8 &a, uint32_t block, bool normed, float scale, float unit, const int8_t *codes, float sc) {
    const uint32_t lane = threadIdx.x & 63u, j = lane & 15u, at = block * 32u + (lane >> 4) * 8u; // this lane's columns
    float x[8];
    uint4 x16;
    float4 u, v;
    if constexpr (BF16) {
        x16 = *(const uint4 *)(a.x_hi + at);
    } else {
        u = *(const float4 *)(a.x + at), v = *(const float4 *)(a.x + at + 4u);
    }
    const uint2 w = *(const uint2 *)(codes + at);
    __builtin_amdgcn_sched_barrier(0); // (both on their way before either is waited for)
    if constexpr (BF16) {
        const uint32_t half[4] = {x16.x, x16.y, x16.z, x16.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) x[2 * e] = __uint_as_float(half[e] << 16), x[2 * e + 1] = __uint_as_float(half[e] & 0xffff0000u);
    } else {
        x[0] = u.x, x[1] = u.y, x[2] = u.z, x[3] = u.w, x[4] = v.x, x[5] = v.y, x[6] = v.z, x[7] = v.w;
        if (normed) {
            const float4 n = *(const float4 *)(a.norm_w + at), m = *(const float4 *)(a.norm_w + at + 4u);
            const float nw[8] = {n.x, n.y, n.z, n.w, m.x, m.y, m.z, m.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = x[e] * scale * nw[e];
        }
    }
    const int32_t shift = 1 - __builtin_amdgcn_frexp_expf(unit);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float rest = Q8Whole::rest(x[e], shift), of_rest = BF16 ? 0.0f : __builtin_truncf(rest);
        const float less = __builtin_amdgcn_ldexpf(rest - of_rest, -(shift + Q8WHOLE_REST));
        const float whole = __builtin_fabsf(Q8Whole::whole(x[e], shift));
        // (all of it: what `whole` may be too small for, what is not finite)
        x[e] = whole >= 1.0f / (float)(1 << Q8WHOLE_REST) && whole <= 0x1p30f ? less : x[e];
    }
    bf16x8 hi, lo;
    q8_split8(x, hi, lo);
    const floatx4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    const floatx4 sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(!BF16 && (j & 1u) ? lo : hi, q8_codes_to_bf16_perm(w), zero4, 0, 0, 0);
    return (BF16 ? sum[0] : sum[0] + sum[1]) * sc;
}

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
// LDS of q8_one_body: the planes of each pair of blocks (and of one more, that the last turn may read and not use), the units, and
// (f32) the planes of the rest.
#define Q8ONE_PAIR 256u // bytes
#define Q8ONE_REST 128u
template <int NW, int REDS = 1> struct Q8OneLds { // (one for all numbers of pairs in flight: each would have its own)
    float red[REDS][NW][64], norm[NW];
    uint32_t finer[NW];
    __attribute__((aligned(16))) uint32_t zero[512]; // what lanes read that hold rows of the other block or pair
};
// U: twos of pairs of blocks a wavefront has in flight, no more than its share: what all wavefronts ask for beyond it costs more
// than it saves in waits. us, with 4 / the smallest that takes the columns in one turn: 16,384 x 512 9.7 / 5.7, x 1,056 7.2 / 6.4,
// x 1,536 10.9 / 8.8, x 2,048 11.0 / 10.0, x 2,560 12.9 / 12.0, 2,880 x 2,048 3.9 / 3.6; past 2,560 columns no gain (16,384 x 2,880
// 11.7 / 11.8), so 4 there: 4,096 columns in one turn of eight wavefronts.
// MANY: the workgroup takes the row tiles blockIdx.x, blockIdx.x + gridDim.x, .. of a.tiles, of all matrices that `a` names, and asks
// for the next one's codes before it puts the sums of one together. (Else one tile, of the matrix that `a` has been made to name.)
template <bool BF16, int NW, bool PREPARE, int U, bool MANY = false>
__device__ __forceinline__ void q8_one_turns(const lng_k_q8 &a, uint32_t tile, char *s_mem, Q8OneLds<NW, MANY ? 2 : 1> &lds, const lng_k_prepare *prepare = nullptr, uint32_t which = 0) {
    constexpr int T = 64 * NW;
    float (&s_norm)[NW] = lds.norm;
    uint32_t (&s_finer)[NW] = lds.finer, (&s_zero)[512] = lds.zero;
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 15u, kg = lane >> 4;
    const uint32_t blocks = a.cols / 32u, pairs = (blocks + 1u) / 2u, chunks = a.cols / 8u, mine = threadIdx.x;
    const uint32_t from = wave * pairs / NW, to = (wave + 1u) * pairs / NW;
    // The tile's rows, the instruction's columns: a.one_rows of them, one after another or (PREPARE: what rotation by halves pairs
    // belongs to one tile) half as many pairs of rows 32 apart, in lanes j and j + 8. The columns past them repeat the last.
    // (a uniform base and 32-bit offsets: a row of the tile is at most 127 x 24,576 bytes on)
    bool row_mine;
    uint32_t row_on, out_row, w_row, w_row_odd, sc_row; // out_row: of the matrix
    const int8_t *w_src;
    const uint16_t *sc_src;
    float *y_dst;
    auto aim = [&](const int8_t *codes, const uint16_t *scales, float *to, uint32_t rows, uint32_t at) {
        if constexpr (PREPARE) {
            const uint32_t half = a.one_rows / 2u, first = at * half, last = (rows / 2u - first < half ? rows / 2u - first : half) - 1u;
            const uint32_t pair = first + ((j & 7u) < last ? j & 7u : last);
            out_row = (pair >> 5) * 64u + (pair & 31u) + (j & 8u) * 4u;
            row_mine = (j & 7u) <= last;
        } else {
            const uint32_t first = at * a.one_rows, last = (rows - first < a.one_rows ? rows - first : a.one_rows) - 1u;
            out_row = first + (j < last ? j : last);
            row_mine = j <= last;
        }
        const uint32_t r0 = __builtin_amdgcn_readfirstlane(out_row);
        row_on = out_row - r0;
        w_src = codes + (uint64_t)r0 * a.cols;
        sc_src = scales + (uint64_t)r0 * blocks;
        w_row = row_on * a.cols + 16u * kg;
        w_row_odd = w_row - ((blocks & 1u) && kg >= 2u ? 32u : 0u);
        sc_row = row_on * blocks;
        y_dst = to;
    };
    auto aim_at = [&](uint32_t id) {
        uint32_t of = 0; // 1 + the one of a.more
#pragma unroll
        for (uint32_t i = 0; i < LNG_Q8_MORE; ++i) of = i < a.n_more && id >= a.more[i].first_tile ? i + 1u : of;
        if (of == 0) {
            aim(a.codes, a.scales, a.y, a.rows, id);
        } else {
            const auto &m = a.more[of - 1u];
            aim(m.codes, m.scales, m.y, m.rows, id - m.first_tile);
        }
    };
    if constexpr (MANY) aim_at(tile);
    else aim(a.codes, a.scales, a.y, a.rows, tile);
    float *s_unit = (float *)(s_mem + (pairs + 1u) * Q8ONE_PAIR);
    char *s_rest = s_mem + ((pairs + 1u) * (Q8ONE_PAIR + 8u) + 15u) / 16u * 16u;

    // A compute unit's loads come back in the order in which its wavefronts ask for them. x (and the weights of its norm) is
    // waited for first, so every wavefront asks for its part before any asks for codes; then the scales, the codes, what is
    // added and prepared at the end. Nothing is waited for before all of it is asked for.
    float x[8], nw[8];
    uint4 x16;
    auto load = [&](uint32_t chunk, const float *src, float (&into)[8]) {
        const float4 u = *(const float4 *)(src + 8u * chunk), v = *(const float4 *)(src + 8u * chunk + 4u);
        into[0] = u.x, into[1] = u.y, into[2] = u.z, into[3] = u.w, into[4] = v.x, into[5] = v.y, into[6] = v.z, into[7] = v.w;
    };
    const bool normed = !BF16 && a.norm_w != nullptr; // uniform
    const uint32_t own = mine < chunks ? mine : chunks - 1u;
    if constexpr (BF16) {
        x16 = *(const uint4 *)(a.x_hi + 8u * own);
    } else {
        load(own, a.x, x);
        if (normed) load(own, a.norm_w, nw);
    }
    uint16_t sc[U];
    uint4 w[2 * U];
    // (Nothing is put in place of what is not loaded: a value merged with another after a branch is copied, and waits. And what
    // is loaded in every case is what the wait for x can count on being behind it: so the first two pairs (past the run: the last
    // one again) and all scales.)
    auto ask = [&](uint32_t base) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t block = 2u * base + 4u * u + kg;
            sc[u] = sc_src[sc_row + (block < blocks ? block : blocks - 1u)];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u == 0 || base + 2u * u < to) { // uniform
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t at = base + 2u * u + h, pair = at < to ? at : to ? to - 1u : 0u;
                    if (h == 0 || (U > 1 && u == 0) || at < to) w[2 * u + h] = *(const uint4 *)(w_src + ((pair == pairs - 1u ? w_row_odd : w_row) + 64u * pair)); // a last pair of one block: the block again
                }
            }
        }
    };
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier(); // (waits for no memory)
    __builtin_amdgcn_sched_barrier(0);
    ask(from);
    const float *any = (const float *)a.codes;
    float bias, held;
    auto ask_added = [&] {
        if constexpr (U > 1) {
            bias = *(a.bias ? a.bias + out_row : any);
            held = *(a.accumulate ? y_dst + out_row : a.residual ? a.residual + out_row : any); // (never both)
        } else {
            if (a.bias) bias = a.bias[out_row];
            if (a.accumulate) held = y_dst[out_row];
            if (a.residual) held = a.residual[out_row];
        }
    };
    ask_added();
    Q8Prepared ready;
    if constexpr (PREPARE) ready.ask<true>(*prepare, which, 0, out_row, any);
    __builtin_amdgcn_sched_barrier(0);

    for (uint32_t i = mine; i < 512u; i += T) s_zero[i] = 0u;
    float scale = 1.0f;
    if (normed) {
        float ss = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
        if (mine >= chunks) ss = 0.0f;
        for (uint32_t c = mine + T; c < chunks; c += T) {
            float more[8];
            load(c, a.x, more);
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += more[e] * more[e];
        }
        ss = wave_sum(ss);
        if (lane == 0) s_norm[wave] = ss;
        __syncthreads();
        float total = 0.0f;
#pragma unroll
        for (int i = 0; i < NW; ++i) total += s_norm[i];
        scale = 1.0f / sqrtf(total / (float)a.cols + a.eps);
    }
    bool finer = false;
    for (uint32_t c = mine; c < chunks; c += T) { // (four chunks to a block, T and the chunks multiples of four: quads of lanes stay together)
        if constexpr (BF16) {
            if (c != mine) x16 = *(const uint4 *)(a.x_hi + 8u * c);
            const uint32_t half[4] = {x16.x, x16.y, x16.z, x16.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) x[2 * e] = __uint_as_float(half[e] << 16), x[2 * e + 1] = __uint_as_float(half[e] & 0xffff0000u);
        } else {
            if (c != mine) {
                load(c, a.x, x);
                if (normed) load(c, a.norm_w, nw);
            }
            if (normed) {
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = x[e] * scale * nw[e];
            }
        }
        Q8Whole whole;
        whole.make<BF16 ? 8 : 18>(x);
        char *put = s_mem + (c >> 3) * Q8ONE_PAIR + (c & 7u) * 8u;
#pragma unroll
        for (int k = 0; k < 4; ++k) *(uint2 *)(put + 64u * k) = whole.plane[k];
        if ((c & 3u) == 0) s_unit[c >> 2] = whole.unit;
        if (whole.unit < 0.0f) {
            if constexpr (BF16) {
                finer = true;
            } else {
                finer |= whole.not_finite || whole.below(26);
                uint2 rest[2];
                whole.make_rest(x, rest);
                put = s_rest + (c >> 3) * Q8ONE_REST + (c & 7u) * 8u;
#pragma unroll
                for (int k = 0; k < 2; ++k) *(uint2 *)(put + 64u * k) = rest[k];
            }
        }
    }
    const bool some_finer = __builtin_amdgcn_ballot_w64(finer) != 0;
    if (lane == 0) s_finer[wave] = some_finer;
    if constexpr (PREPARE) ready.place<true>(*prepare, which, 0, out_row);
    __syncthreads();

    const uint32_t some = s_finer[lane & (NW - 1u)];
    const i32x4 zero = {0, 0, 0, 0};
    const bool block_mine = ((j >> 2) & 1u) == (kg >> 1);
    for (uint32_t round = 0;; ++round) { // (!MANY: once)
        float y = 0.0f;
        for (uint32_t base = from; base < to; base += 2u * U) {
            if (base != from) ask(base);
            const char *planes = s_mem + base * Q8ONE_PAIR + (j & 3u) * 64u + 16u * kg;
            const char *first = block_mine && j < 8u ? planes : (const char *)s_zero;
            const char *second = block_mine && j >= 8u ? planes + Q8ONE_PAIR : (const char *)s_zero;
            i32x4 p[2 * U];
            float unit[U];
    #pragma unroll
            for (int u = 0; u < U; ++u) {
                if (u == 0 || base + 2u * u < to) {
                    p[2 * u] = *(const i32x4 *)(first + 2u * u * Q8ONE_PAIR);
                    p[2 * u + 1] = *(const i32x4 *)(second + 2u * u * Q8ONE_PAIR);
                    unit[u] = s_unit[2u * base + 4u * u + kg];
                }
            }
    #pragma unroll
            for (int u = 0; u < U; ++u) {
                if (u == 0 || base + 2u * u < to) {
                    i32x4 acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(p[2 * u], __builtin_bit_cast(i32x4, w[2 * u]), zero, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(p[2 * u + 1], __builtin_bit_cast(i32x4, w[2 * u + 1]), acc, 0, 0, 0);
                    float sum = __builtin_fmaf((float)acc[3], 256.0f, (float)acc[2]);
                    sum = __builtin_fmaf(sum, 256.0f, (float)acc[1]);
                    sum = __builtin_fmaf(sum, 256.0f, (float)acc[0]);
                    const uint32_t block = 2u * base + 4u * u + kg;
                    const bool used = block < 2u * to && block < blocks;
                    if constexpr (!BF16) {
                        if (__builtin_amdgcn_ballot_w64(used && unit[u] < 0.0f)) {
                            const char *rest = s_rest + (base + 2u * u) * Q8ONE_REST + (j & 3u) * 64u + 16u * kg;
                            const i32x4 r0 = *(const i32x4 *)(block_mine && (j & 3u) < 2u && j < 8u ? rest : (const char *)s_zero);
                            const i32x4 r1 = *(const i32x4 *)(block_mine && (j & 3u) < 2u && j >= 8u ? rest + Q8ONE_REST : (const char *)s_zero);
                            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(r0, __builtin_bit_cast(i32x4, w[2 * u]), zero, 0, 0, 0);
                            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(r1, __builtin_bit_cast(i32x4, w[2 * u + 1]), acc, 0, 0, 0);
                            const float more = __builtin_fmaf((float)acc[1], 256.0f, (float)acc[0]);
                            if (unit[u] < 0.0f) sum = __builtin_fmaf(more, 1.0f / (float)(1 << Q8WHOLE_REST), sum);
                        }
                    }
                    const float next = __builtin_fmaf(sum * f16_bits_to_f32(sc[u]), __builtin_fabsf(unit[u]), y);
                    y = used ? next : y;
                }
            }
        }
        if (__builtin_amdgcn_ballot_w64(some != 0u)) { // uniform in the workgroup
            for (uint32_t b = 2u * from; b < 2u * to; b += 64u) {
                const bool more = b + lane < 2u * to && b + lane < blocks && s_unit[b + lane] < 0.0f;
                for (uint64_t left = __builtin_amdgcn_ballot_w64(more); left; left &= left - 1u) {
                    const uint32_t block = b + (uint32_t)__builtin_ctzll(left);
                    const float rest = q8_one_rest<BF16>(a, block, normed, scale, -s_unit[block], w_src + row_on * a.cols, f16_bits_to_f32(sc_src[sc_row + block]));
                    if (kg == 0) y += rest;
                }
            }
        }
        float (&s_red)[NW][64] = lds.red[MANY ? round & 1u : 0u]; // (in turn: one may still be read when the other is written)
        float *const to_y = y_dst;
        const uint32_t to_row = out_row;
        const bool writes = lane < 16u && row_mine;
        const float bias_now = bias, held_now = held;
        const bool again = MANY && tile + gridDim.x < a.tiles; // uniform
        if constexpr (MANY) {
            if (again) {
                tile += gridDim.x;
                aim_at(tile);
                ask(from);
                ask_added();
            }
        }
        s_red[wave][lane] = y;
        __syncthreads();
        if (wave == (MANY ? round % NW : 0u)) {
            float sum = 0.0f;
#pragma unroll
            for (int i = 0; i < NW; ++i) sum += s_red[i][lane];
            const auto s16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(sum), __float_as_uint(sum), false, false);
            sum = __uint_as_float(s16[0]) + __uint_as_float(s16[1]);
            const auto s32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(sum), __float_as_uint(sum), false, false);
            sum = __uint_as_float(s32[0]) + __uint_as_float(s32[1]);
            if (a.bias) sum = sum + bias_now;
            if (a.accumulate) sum = held_now + sum;
            if (writes) {
                to_y[to_row] = sum;
                if (a.residual) a.residual[to_row] = held_now + sum;
                if constexpr (PREPARE) {
                    const float there = __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(sum), 0x128, 0xf, 0xf, true)); // row_ror:8, 32 rows away
                    ready.store(*prepare, which, to_row, sum, there);
                }
            }
        }
        if (!again) return;
    }
}

template <bool BF16, int NW, bool PREPARE = false>
__device__ __forceinline__ void q8_one_body(const lng_k_q8 &a, uint32_t tile, char *s_mem, const lng_k_prepare *prepare = nullptr, uint32_t which = 0) {
    __shared__ Q8OneLds<NW> lds;
    if (a.cols <= 128u * NW) q8_one_turns<BF16, NW, PREPARE, 1>(a, tile, s_mem, lds, prepare, which);
    else if (a.cols <= 256u * NW) q8_one_turns<BF16, NW, PREPARE, 2>(a, tile, s_mem, lds, prepare, which);
    else if (a.cols <= 320u * NW) q8_one_turns<BF16, NW, PREPARE, 3>(a, tile, s_mem, lds, prepare, which);
    else q8_one_turns<BF16, NW, PREPARE, 4>(a, tile, s_mem, lds, prepare, which);
}

// One position of more tiles than the device holds workgroups of. When each tile was a workgroup, the planes of x were made for
// every one of them, 1 us that the codes of the next did not hide. us, f32 positions, the kernel before the integer one / a tile a
// workgroup / so: 16,384 x 512 5.6 / 5.4 / 5.2, 65,536 x 1,024 20.4 / 22.0 / 15.4, x 2,880 35.7 / 37.5 / 35.2, x 4,096 50.0 / 55.7 / 50.5;
// with the norm 6.7 / 6.6 / 5.9, 23.8 / 28.1 / 16.2, 39.2 / 43.2 / 35.5, 52.0 / 60.7 / 51.3. 150,000 x 4,096 105 / 119 / 109, x 2,880 74.5 / 79.1 /
// 76.3 (with the norm 109 / 130 / 110, 81 / 93 / 77).
// As many tiles to each workgroup, one grid apart: a run of neighbours to each is 5 to 8 % slower, workgroups of 2 to 9 tiles each up
// to 45 %. Three twos of pairs in flight where they are all of a turn (24,576 x 2,880 16.7 with two, 15.3); more (9 % slower at
// 4,096 columns, and f32 keeps registers in memory) or a third workgroup in a unit (1 % slower) read no faster.
template <bool BF16, int NW>
__device__ __forceinline__ void q8_tall_body(const lng_k_q8 &a, char *s_mem) {
    __shared__ Q8OneLds<NW, 2> lds;
    if (a.cols <= 128u * NW) q8_one_turns<BF16, NW, false, 1, true>(a, blockIdx.x, s_mem, lds);
    else if (a.cols <= 256u * NW || a.cols > 384u * NW) q8_one_turns<BF16, NW, false, 2, true>(a, blockIdx.x, s_mem, lds);
    else q8_one_turns<BF16, NW, false, 3, true>(a, blockIdx.x, s_mem, lds);
}

// 2 to 16 f32 positions of 2,048 to 4,096 columns in one dispatch, with the RMS norm if norm_w is set: x goes through the matrix
// unit as it is (times the norm's weights), its squares are added up on the way and each position's scale multiplies the result (as
// exact as normalising it first: two bf16 values hold as much of a number at any size).
// So there is no dispatch of planes before it and x is read once: eight lanes to a position's 128 bytes of a block, split, and
// turned into operand order through LDS that only this wavefront uses. x is most of what a workgroup reads (16 positions of 2,880
// columns: 184 KB beside 46 KB of codes for 16 rows), so a workgroup takes up to 32 rows, NT runs of 16, and has a compute unit
// to itself: all its loads of a turn but the last pairs' x are on their way at once.
// With planes made by a dispatch before it and tiles of 16 rows / so, us, 16 positions: 5,120 x 2,880 12.4 / 10.9 with the norm,
// 11.9 / 11.1 without, 4,112 x 4,096 15.7 / 13.1 and 15.1 / 13.4, 8,192 x 2,048 11.3 / 10.6 and 10.7 / 10.4; in a decoding step of
// sixteen sequences (kernel trace, preparation included) 4.7 + 11.4 / 13.0 to 13.5. As many rows as have a unit each with one workgroup
// of 16 gain nothing (2,880 x 4,096 10.9 / 10.8).
// U: pairs of blocks of a wavefront (2,880 columns: five or six of 6; up to 4,096: 8).
template <int U, bool PREPARE>
__device__ __forceinline__ void q8_few_split_turn(const lng_k_q8 &a, uint32_t tile, char *s_mem, const lng_k_prepare *prepare = nullptr, uint32_t which = 0) {
    constexpr int NW = 8, NT = 2, D = 2; // D: pairs of x in flight (3: 2 % slower, 6: 8 %)
    constexpr uint32_t STRIDE = 80, PLANE = 16 * STRIDE;
    __shared__ float s_red[NW][NT * 4][64];
    __shared__ float s_ss[NW][16];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = lane & 15u, kg = lane >> 4;
    const uint32_t blocks = a.cols / 32u, pairs = (blocks + 1u) / 2u, from = wave * pairs / NW, to = (wave + 1u) * pairs / NW, words = pairs | 1u;
    char *s_x = s_mem + wave * 4u * PLANE; // [block of a pair][plane][position]
    uint32_t *s_sc = (uint32_t *)(s_mem + NW * 4u * PLANE);
    // the tile's row k of 16 NT (see q8_one_turns), those past its last the last again
    const uint32_t first = tile * (PREPARE ? a.one_rows / 2u : a.one_rows), rows = PREPARE ? a.rows / 2u : a.rows;
    const uint32_t last = (rows - first < (PREPARE ? a.one_rows / 2u : a.one_rows) ? rows - first : (PREPARE ? a.one_rows / 2u : a.one_rows)) - 1u;
    auto row_of = [&](uint32_t k) {
        if constexpr (PREPARE) {
            const uint32_t at = (k >> 4) * 8u + (k & 7u), pair = first + (at < last ? at : last);
            return (pair >> 5) * 64u + (pair & 31u) + (k & 8u) * 4u;
        } else {
            return first + (k < last ? k : last);
        }
    };
    auto has_row = [&](uint32_t k) { return (PREPARE ? (k >> 4) * 8u + (k & 7u) : k) <= last; };
    const uint32_t r0 = row_of(0);
    const int8_t *w_src = a.codes + (uint64_t)r0 * a.cols; // (uniform bases and 32-bit offsets, as in q8_one_turns)
    const uint16_t *sc_src = a.scales + (uint64_t)r0 * blocks;
    uint32_t w_row[NT], w_row_odd[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        w_row[nt] = (row_of(16u * nt + j) - r0) * a.cols + 16u * kg;
        w_row_odd[nt] = w_row[nt] - ((blocks & 1u) && kg >= 2u ? 32u : 0u);
    }
    // this thread's output: accumulator register wave % 4 of run wave / 4
    const uint32_t out_p = 4u * kg + (wave & 3u), out_k = 16u * (wave >> 2) + j, out_row = row_of(out_k);
    const bool mine = wave < 4u * NT && out_p < a.n && has_row(out_k);
    const uint32_t some_p = out_p < a.n ? out_p : a.n - 1u;

    // What is asked for first comes first. The preparation's items (their table's rows are asked for once x is here), the scales,
    // x, the codes.
    lng_prepare_item it;
    if constexpr (PREPARE) {
        if (prepare->items) it = prepare->items[some_p];
    }
    const bool whole_words = (((uintptr_t)sc_src & 3u) | (blocks & 1u)) == 0; // uniform
    uint32_t sc_now[2 * NT], sc_then[2 * NT];
    auto sc_row = [&](int i) { return (row_of(wave * 2u * NT + i) - r0) * blocks; }; // (scalar)
    {
        const uint32_t at = lane < pairs ? lane : pairs - 1u; // (at most 64 pairs)
#pragma unroll
        for (int i = 0; i < 2 * NT; ++i) {
            const uint16_t *src = sc_src + sc_row(i) + 2u * at;
            if (whole_words) {
                sc_now[i] = *(const uint32_t *)src;
            } else {
                sc_now[i] = src[0];
                sc_then[i] = src[2u * at + 1u < blocks ? 1 : 0];
            }
        }
    }
    const float *x_src[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t p = 8u * h + (lane >> 3);
        x_src[h] = a.x + (uint64_t)(p < a.n ? p : a.n - 1u) * a.x_stride + 4u * (lane & 7u);
    }
    const bool normed = a.norm_w != nullptr; // uniform
    const float *nw_src = (normed ? a.norm_w : a.x) + 4u * (lane & 7u);
    float4 x[D][2][2], nw[D][2]; // [pair][block][positions 0-7, 8-15]
    // (A pair past the run loads its first again and is not used: nothing is loaded behind a branch, so every wait knows what is
    // behind what it waits for.)
    auto pair_of = [&](uint32_t u) { return from + u < to ? from + u : from; };
    auto ask_x = [&](uint32_t pair, float4 (&into)[2][2], float4 (&weights)[2]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t b = 2u * pair + h < blocks ? 2u * pair + h : blocks - 1u;
            into[h][0] = *(const float4 *)(x_src[0] + 32u * b);
            into[h][1] = *(const float4 *)(x_src[1] + 32u * b);
            weights[h] = *(const float4 *)(nw_src + 32u * b);
        }
    };
    uint4 w[U][NT];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d < D; ++d) ask_x(pair_of(d), x[d], nw[d]);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier(); // every wavefront's x before any one's codes; waits for no memory
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t pair = pair_of(u);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) w[u][nt] = *(const uint4 *)(w_src + ((pair == pairs - 1u ? w_row_odd[nt] : w_row[nt]) + 64u * pair));
    }
    const float *any = (const float *)a.codes;
    const float bias = *(a.bias ? a.bias + out_row : any);
    float *yp = a.y + (uint64_t)some_p * a.y_stride + out_row, *res = a.residual + (uint64_t)some_p * a.rows + out_row;
    const float held = *(a.accumulate ? yp : a.residual ? res : any); // (never both)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i) {
        uint32_t *to_row = s_sc + (wave * 2u * NT + i) * words;
        const uint32_t both = whole_words ? sc_now[i] : __builtin_amdgcn_perm(sc_then[i], sc_now[i], 0x05040100u);
        if (lane < pairs) to_row[lane] = both;
    }
    __syncthreads();
    Q8Prepared ready;
    if constexpr (PREPARE) {
        lng_prepare_item one = prepare->first;
        if (prepare->items) one = it;
        ready.ask_of(*prepare, which, one, prepare->items ? 0u : some_p, out_row, any);
        ready.place_of(*prepare, which, one, prepare->items ? 0u : some_p, out_row);
    }

    floatx4 y[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) y[nt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    const floatx4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    float ss[2] = {0.0f, 0.0f};
    const uint32_t put = (lane >> 3) * STRIDE + 8u * (lane & 7u), get = j * STRIDE + 16u * q8_mid_chunk(kg);
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint32_t pair = from + u;
        if (pair < to) { // uniform
            const bool second = 2u * pair + 1u < blocks; // uniform
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    const float4 v = x[u % D][h][g], n = nw[u % D][h];
                    float e[4] = {v.x, v.y, v.z, v.w};
                    if (h == 0 || second) ss[g] += e[0] * e[0] + e[1] * e[1] + e[2] * e[2] + e[3] * e[3];
                    if (normed) e[0] *= n.x, e[1] *= n.y, e[2] *= n.z, e[3] *= n.w;
                    bf16x4 hi, lo;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const __bf16 top = (__bf16)e[i];
                        hi[i] = top;
                        lo[i] = (__bf16)(e[i] - (float)top);
                    }
                    *(bf16x4 *)(s_x + (2 * h) * PLANE + 8 * g * STRIDE + put) = hi;
                    *(bf16x4 *)(s_x + (2 * h + 1) * PLANE + 8 * g * STRIDE + put) = lo;
                }
            }
            bf16x8 op[2][2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                op[h][0] = as_bf16x8(*(const uint4 *)(s_x + (2 * h) * PLANE + get));
                op[h][1] = as_bf16x8(*(const uint4 *)(s_x + (2 * h + 1) * PLANE + get));
            }
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const auto s0 = __builtin_amdgcn_permlane32_swap(w[u][nt].x, w[u][nt].z, false, false);
                const auto s1 = __builtin_amdgcn_permlane32_swap(w[u][nt].y, w[u][nt].w, false, false);
                const bf16x8 b0 = q8_codes_to_bf16_perm(make_uint2(s0[0], s1[0])), b1 = q8_codes_to_bf16_perm(make_uint2(s0[1], s1[1]));
                const uint32_t both = s_sc[(16u * nt + j) * words + pair];
                const float c0 = f16_bits_to_f32((uint16_t)both), c1 = f16_bits_to_f32((uint16_t)(both >> 16));
                floatx4 p0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op[0][0], b0, zero4, 0, 0, 0);
                floatx4 p1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op[1][0], b1, zero4, 0, 0, 0);
                p0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op[0][1], b0, p0, 0, 0, 0);
                p1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op[1][1], b1, p1, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i) y[nt][i] = __builtin_fmaf(c0, p0[i], y[nt][i]);
                if (second) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) y[nt][i] = __builtin_fmaf(c1, p1[i], y[nt][i]);
                }
            }
        }
        if (u + D < U) {
            __builtin_amdgcn_sched_barrier(0);
            ask_x(pair_of(u + D), x[u % D], nw[u % D]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int g = 0; g < 2; ++g) { // over the eight lanes of a position
        auto across = [&](auto ctrl) { ss[g] += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(ss[g]), decltype(ctrl)::value, 0xf, 0xf, true)); };
        across(std::integral_constant<int, 0xB1>{});  // quad_perm [1,0,3,2]
        across(std::integral_constant<int, 0x4E>{});  // quad_perm [2,3,0,1]
        across(std::integral_constant<int, 0x141>{}); // row_half_mirror
        if ((lane & 7u) == 0) s_ss[wave][8u * g + (lane >> 3)] = ss[g];
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) s_red[wave][4 * nt + i][lane] = y[nt][i];
    }
    __syncthreads();
    if (wave >= 4u * NT) return;
    float sum = 0.0f, squares = 0.0f;
#pragma unroll
    for (int i = 0; i < NW; ++i) sum += s_red[i][wave][lane], squares += s_ss[i][out_p];
    if (normed) sum = sum * (1.0f / sqrtf(squares / (float)a.cols + a.eps));
    if (a.bias) sum = sum + bias;
    if (a.accumulate) sum = held + sum;
    float there = 0.0f;
    if constexpr (PREPARE) there = __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(sum), 0x128, 0xf, 0xf, true)); // row_ror:8, 32 rows away
    if (!mine) return;
    *yp = sum;
    if (a.residual) *res = held + sum;
    if constexpr (PREPARE) ready.store(*prepare, which, out_row, sum, there);
}

#define Q8_FEW(name, body, what, nw) \
    extern "C" __global__ __launch_bounds__(64 * nw, nw / 2) void name(lng_k_q8 a) { \
        extern __shared__ __attribute__((aligned(16))) char s_mem[]; /* as many bytes as q8_record_few works out */ \
        const uint32_t tile = q8_select_matrix(a); \
        body<what, nw>(a, tile, s_mem); \
    }
Q8_FEW(lng_q8_few, q8_few_body, Q8F_PLANES, 8)
Q8_FEW(lng_q8_few_bf16, q8_few_body, Q8F_BF16, 8)
Q8_FEW(lng_q8_few_f32, q8_few_body, Q8F_F32, 8)
Q8_FEW(lng_q8_one, q8_one_body, false, 8)
Q8_FEW(lng_q8_one_bf16, q8_one_body, true, 8)

#define Q8_TALL(name, bf16, nw) \
    extern "C" __global__ __launch_bounds__(64 * nw, nw / 2) void name(lng_k_q8 a) { \
        extern __shared__ __attribute__((aligned(16))) char s_mem[]; \
        q8_tall_body<bf16, nw>(a, s_mem); \
    }
Q8_TALL(lng_q8_tall, false, 8)
Q8_TALL(lng_q8_tall_bf16, true, 8)

// q, k and v with the preparation of attention after them.
#define Q8_FEW_PREPARE(name, body, what, nw) \
    extern "C" __global__ __launch_bounds__(64 * nw, nw / 2) void name(lng_k_q8_prepare both) { \
        extern __shared__ __attribute__((aligned(16))) char s_mem[]; \
        lng_k_q8 a = both.q8; \
        const uint32_t which = blockIdx.x >= a.more[1].first_tile ? 2u : blockIdx.x >= a.more[0].first_tile ? 1u : 0u; \
        const uint32_t tile = q8_select_matrix(a); \
        body<what, nw, true>(a, tile, s_mem, &both.prepare, which); \
    }
Q8_FEW_PREPARE(lng_q8_few_prepare, q8_few_body, Q8F_PLANES, 8)
Q8_FEW_PREPARE(lng_q8_few_f32_prepare, q8_few_body, Q8F_F32, 8)
Q8_FEW_PREPARE(lng_q8_one_prepare, q8_one_body, false, 8)

template <bool PREPARE = false>
__device__ __forceinline__ void q8_few_split_body(const lng_k_q8 &a, uint32_t tile, char *s_mem, const lng_k_prepare *prepare = nullptr, uint32_t which = 0) {
    if (a.cols <= 3072u) q8_few_split_turn<6, PREPARE>(a, tile, s_mem, prepare, which);
    else q8_few_split_turn<8, PREPARE>(a, tile, s_mem, prepare, which);
}

extern "C" __global__ __launch_bounds__(512, 2) void lng_q8_few_split(lng_k_q8 a) {
    extern __shared__ __attribute__((aligned(16))) char s_mem[];
    const uint32_t tile = q8_select_matrix(a);
    q8_few_split_body(a, tile, s_mem);
}
extern "C" __global__ __launch_bounds__(512, 2) void lng_q8_few_split_prepare(lng_k_q8_prepare both) {
    extern __shared__ __attribute__((aligned(16))) char s_mem[];
    lng_k_q8 a = both.q8;
    const uint32_t which = blockIdx.x >= a.more[1].first_tile ? 2u : blockIdx.x >= a.more[0].first_tile ? 1u : 0u;
    const uint32_t tile = q8_select_matrix(a);
    q8_few_split_body<true>(a, tile, s_mem, &both.prepare, which);
}
