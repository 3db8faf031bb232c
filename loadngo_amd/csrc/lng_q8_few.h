// Q8_0 products of fewer than 32 positions (17 to 31 of matrices of many rows share lng_q8_mid's tiles): lng_q8_norm_frag,
// lng_q8_few*, lng_q8_one*. (Included by lng_kernels.hip after lng_q8_mid.h; see there for how a product goes through the matrix unit.)

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
    __device__ __forceinline__ void ask(const lng_k_prepare &p, uint32_t which, uint32_t position, uint32_t row) {
        const lng_prepare_item it = p.items ? p.items[position] : p.first;
        const uint32_t r = p.items ? 0u : position; // a table's items are of one position each
        const float *b = which == 0 ? p.q_bias : which == 1 ? p.k_bias : p.v_bias;
        bias = b ? b[row] : 0.0f;
        bias_there = b && which < 2u ? b[row ^ 32u] : 0.0f;
        c = 0.0f, s = 0.0f;
        if (which < 2u) {
            const float2 t = *(const float2 *)(p.table + it.table_offset + ((uint64_t)r * 32u + (row & 31u)) * 8u);
            c = t.x, s = t.y;
        }
        const uint32_t es = p.out_dtype == LNG_BF16 ? 2u : 4u;
        if (which == 0) {
            to = p.q_out + it.q_out_offset + ((uint64_t)r * p.heads * 64u + row) * es;
        } else {
            const uint64_t at = ((it.start + r) % it.slots * p.kv_heads * 64u + row) * es;
            to = which == 1 ? p.k_cache + it.k_cache_offset + at : p.v_cache + it.v_cache_offset + at;
        }
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
// matrix: 5,120 x 2,880 (q, k and v, 15.7 MB) with the norm, in a batch of 16 such: 1 position 7.8 us (11.1 when every
// wavefront asked for half of its blocks at a time and split x for each), 2 to 16: 12 us with the planes' dispatch (20-27
// when each workgroup normalised and split all positions itself), 31: 14 us (38); 2,880 x 4,096 with bias and residual from
// bf16 1, 16, 31 positions: 6.7, 8.1, 10 us (9.1, 13, 23), from f32 6.9, 11, 16 (11, 19, 35).
// One position with every load of a turn really on its way before the first is waited for: 16,384 x 2,880 14.9 -> 11.7 us
// (bf16 14.3 -> 11.3), 2,048 rows 6.0 -> 5.1 (5.8 -> 4.7).
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
        if (mine) ready.ask(*prepare, which, out_p, out_row);
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

// One position. Its operand planes are made once per workgroup (normalised, split: a thread takes eight columns) and wait
// in LDS. f32: even rows of the A operand are the hi plane, odd ones the lo plane, and one matrix instruction multiplies
// a block by both; all rows of bf16 are the position.
template <bool BF16, int NW, bool PREPARE = false>
__device__ __forceinline__ void q8_one_body(const lng_k_q8 &a, uint32_t tile, char *s_mem, const lng_k_prepare *prepare = nullptr, uint32_t which = 0) {
    constexpr int U = Q8Few<NW>::U, T = 64 * NW;
    __shared__ float s_red[NW][16];
    __shared__ float s_norm[NW];
    Q8Few<NW, PREPARE> m(a, tile, (uint32_t *)(s_mem + (uint64_t)a.cols * (BF16 ? 2u : 4u)));
    const uint32_t chunks = a.cols / 8u, mine = threadIdx.x, out_row = q8_tile_row<PREPARE>(tile) + q8_row_in<PREPARE>(mine & 15u);
    const bool writes = mine < m.rows_here;
    uint4 *s_x = (uint4 *)s_mem; // [plane][chunk of eight columns]
    float x[8] = {}, nw[8] = {};
    uint4 x16 = make_uint4(0, 0, 0, 0);
    auto load = [&](uint32_t chunk, const float *src, float (&to)[8]) {
        const float4 u = *(const float4 *)(src + 8u * chunk), v = *(const float4 *)(src + 8u * chunk + 4u);
        to[0] = u.x, to[1] = u.y, to[2] = u.z, to[3] = u.w, to[4] = v.x, to[5] = v.y, to[6] = v.z, to[7] = v.w;
    };
    const bool normed = !BF16 && a.norm_w != nullptr; // uniform
    if (mine < chunks) {
        if constexpr (BF16) {
            x16 = *(const uint4 *)(a.x_hi + 8u * mine);
        } else {
            load(mine, a.x, x);
            if (normed) load(mine, a.norm_w, nw);
        }
    }
    m.ask_scales();
    float bias = 0.0f, held = 0.0f;
    if (writes && a.bias) bias = a.bias[out_row];
    if (writes && a.accumulate) held = a.y[out_row];
    if (writes && a.residual) held = a.residual[out_row]; // (never with accumulate)
    Q8Prepared ready;
    if constexpr (PREPARE) {
        if (writes) ready.ask(*prepare, which, 0, out_row);
    }
    __builtin_amdgcn_sched_barrier(0);
    m.ask_codes(m.from); // after what is waited for first: loads come back in order
    __builtin_amdgcn_sched_barrier(0);
    m.stage_scales();
    if constexpr (BF16) {
        if (mine < chunks) s_x[mine] = x16;
        for (uint32_t c = mine + T; c < chunks; c += T) s_x[c] = *(const uint4 *)(a.x_hi + 8u * c);
    } else {
        float scale = 0.0f;
        if (normed) {
            float ss = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += x[e] * x[e]; // zeros past the last chunk
            for (uint32_t c = mine + T; c < chunks; c += T) {
                float more[8];
                load(c, a.x, more);
#pragma unroll
                for (int e = 0; e < 8; ++e) ss += more[e] * more[e];
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
            if (m.lane == 0) s_norm[m.wave] = ss;
            __syncthreads();
            float total = 0.0f;
#pragma unroll
            for (int w = 0; w < NW; ++w) total += s_norm[w];
            scale = 1.0f / sqrtf(total / (float)a.cols + a.eps);
        }
        for (uint32_t c = mine; c < chunks; c += T) {
            if (c != mine) {
                load(c, a.x, x);
                if (normed) load(c, a.norm_w, nw);
            }
            if (normed) {
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = x[e] * scale * nw[e];
            }
            bf16x8 hi, lo;
            q8_split8(x, hi, lo);
            s_x[c] = __builtin_bit_cast(uint4, hi);
            s_x[chunks + c] = __builtin_bit_cast(uint4, lo);
        }
    }
    __syncthreads();
    const uint4 *x_at = s_x + q8_mid_chunk(m.kg) + (!BF16 && (m.j & 1u) ? chunks : 0u);
    float y[2] = {0.0f, 0.0f};
    const floatx4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t base = m.from; base < m.to; base += U) {
        if (base != m.from) m.ask_codes(base);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (base + u < m.to) {
                bf16x8 b[2];
                float sc[2];
                m.operands(u, base + u, b, sc);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t block = 2u * (base + u) + h;
                    if (h == 0 || block < m.blocks) { // uniform
                        const floatx4 acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(x_at[4u * block]), b[h], zero4, 0, 0, 0);
                        y[0] = __builtin_fmaf(sc[h], acc[0], y[0]);
                        if constexpr (!BF16) y[1] = __builtin_fmaf(sc[h], acc[1], y[1]);
                    }
                }
            }
        }
    }
    if (m.lane < 16u) s_red[m.wave][m.lane] = y[0] + y[1];
    __syncthreads();
    if (!writes) return;
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) sum += s_red[w][mine];
    if (a.bias) sum = sum + bias;
    if (a.accumulate) sum = held + sum;
    a.y[out_row] = sum;
    if (a.residual) a.residual[out_row] = held + sum;
    if constexpr (PREPARE) ready.store(*prepare, which, out_row, sum, __shfl_xor(sum, 8, 64));
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
