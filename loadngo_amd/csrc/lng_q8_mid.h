// Q8_0 products of a chunk of positions: lng_q8_frag_x, lng_q8_mid*. (Included by lng_kernels.hip; see there
// for how a product goes through the matrix unit.)

// The 16 bytes of columns that lane group kg = lane / 16 of an operand holds of a block, in the order of lng_q8_mid.
__device__ __forceinline__ uint32_t q8_mid_chunk(uint32_t kg) { return (kg & 1u) * 2u + (kg >> 1); }

// x[n][x_stride] f32 as the A operands of lng_q8_mid: hi and lo planes (hi + lo = x to 16 bits) in the order in which a
// wavefront loads them. Group g of 16 positions, block b, plane: 64 lanes x 8 values, lane l = position l % 16, columns
// 8 * q8_mid_chunk(l / 16) .. + 7 of the block. Rows past n are zero.
extern "C" __global__ __launch_bounds__(256) void lng_q8_frag_x(lng_k_q8_split a) {
    const uint32_t blocks = a.cols / 32u;
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    const uint32_t lane = idx & 63u, unit = idx >> 6; // unit = group * blocks + block
    if (unit >= a.n_pad / 16u * blocks) return;
    const uint32_t group = unit / blocks, b = unit - group * blocks;
    const uint32_t p = group * 16u + (lane & 15u);
    float x[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (p < a.n) {
        const float *src = a.x + (uint64_t)p * a.x_stride + 32u * b + 8u * q8_mid_chunk(lane >> 4);
        const float4 u = *(const float4 *)src, v = *(const float4 *)(src + 4);
        x[0] = u.x, x[1] = u.y, x[2] = u.z, x[3] = u.w, x[4] = v.x, x[5] = v.y, x[6] = v.z, x[7] = v.w;
    }
    bf16x8 hi, lo;
    q8_split8(x, hi, lo);
    uint4 *to = (uint4 *)a.hi + (uint64_t)unit * 128u + lane;
    to[0] = __builtin_bit_cast(uint4, hi);
    to[64] = __builtin_bit_cast(uint4, lo);
}

// A workgroup takes 16 NT rows x 16 MT positions and its NW wavefronts share the COLUMNS: each multiplies the whole tile
// over its run of block pairs and the partial results meet in LDS at the end. There is no barrier in the loop, and a
// product of few positions is cut into enough pieces to fill the device: lng_q8_tiled, whose tiles of 256 x 128 walk all
// columns in sequence, takes 88 us for 2,880 columns (125 for 4,096) whatever the rows and positions below 512.
// Bound by what the tiles read through L2 (the positions once per row tile, 64 rows x 64 positions: 10 KB a block of 32
// columns) and, for few positions, by latencies: a start of 3 us, the loads' round trips, the partials' way through LDS.
// Measured, split of x included (q, k and v of 5,120 x 2,880 as one dispatch / 2,880 x 4,096 from bf16; before: three
// products of lng_q8_tiled / one): 32 positions 12 / 8.7 us (275 / 86), 77: 19 / 17 (276 / 87), 512: 57 / 41 (285 / 89),
// 1,024: 94-102 / 62-65 (294 / 89). Two workgroups of four wavefronts per compute unit against one of eight: one's start
// and end under the other's products (512 positions 69 -> 57 us, 1,024: 124 -> 94); the smallest tiles need the eight
// (few workgroups: every wavefront's loads count).
// Codes: a lane loads 16 of a row at once (two blocks: lanes 0-31 the first, 32-63 the second); one swap of register
// halves makes of that the B operands of both blocks, whose columns then come in the order q8_mid_chunk gives.
// bf16 positions are loaded four lanes to a position's 64 bytes (neighbouring lanes in different rows make every lane a
// memory access of its own: 512 positions 58 us against 47) and turned through LDS that only this wavefront uses, rows
// 80 bytes apart: neither the 16-byte stores nor the operand reads of 16 rows meet in a bank. The same for the codes
// costs more in LDS round trips than it saves.
template <int NT, int MT, int PLANES, int NW>
__device__ __forceinline__ void q8_mid_body(const lng_k_q8 &a, uint32_t row_tile, uint32_t pos_tile, char *s_mem) {
    constexpr uint32_t STRIDE = 80;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t j = lane & 15u, kg = lane >> 4;
    const uint32_t r0 = row_tile * 16u * NT, p0 = pos_tile * 16u * MT;
    const uint32_t blocks = a.cols / 32u;
    char *s_x = s_mem + wave * 16u * STRIDE * MT;
    uint16_t *s_sc = (uint16_t *)(s_mem + (PLANES == 1 ? NW * 16u * STRIDE * MT : 0u));
    const uint32_t rows_here = a.rows - r0 < 16u * NT ? a.rows - r0 : 16u * NT;
    const uint32_t put = (lane >> 2) * STRIDE + 16u * (lane & 3u); // where a lane's 16 loaded bytes of x go
    const uint32_t get = j * STRIDE + 16u * q8_mid_chunk(kg);

    const int8_t *w_src[NT];
    uint32_t s_row[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const uint32_t row = 16u * nt + j < rows_here ? 16u * nt + j : rows_here - 1u;
        w_src[nt] = a.codes + (uint64_t)(r0 + row) * a.cols + 16u * kg;
        s_row[nt] = row * blocks;
    }
    const uint16_t *sc_src = a.scales + (uint64_t)r0 * blocks;
    const uint16_t *x_src[MT]; // PLANES == 1: the position this lane loads of each group
    if constexpr (PLANES == 1) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const uint32_t at = p0 + 16u * mt + (lane >> 2), p = at < a.n ? at : a.n - 1u;
            x_src[mt] = a.x_hi + (uint64_t)p * a.plane_stride + 8u * (lane & 3u);
        }
    }
    const uint4 *x_frag = (const uint4 *)a.x_hi; // PLANES == 2: lng_q8_frag_x's layout
    auto load_x = [&](uint32_t b, uint4 (&x)[MT][PLANES]) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            if constexpr (PLANES == 1) {
                x[mt][0] = *(const uint4 *)(x_src[mt] + 32u * b);
            } else {
                const uint4 *at = x_frag + ((uint64_t)(pos_tile * MT + mt) * blocks + b) * 128u;
                x[mt][0] = at[lane];
                x[mt][1] = at[64u + lane];
            }
        }
    };
    auto load_w = [&](uint32_t pair, uint4 (&w)[NT]) {
        // a last pair of one block: its upper lanes load the block again
        const int32_t col = (int32_t)(64u * pair) - (2u * pair + 1u == blocks && kg >= 2u ? 32 : 0); // -32 in the only pair of one block
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) w[nt] = *(const uint4 *)(w_src[nt] + col);
    };

    floatx4 y[NT][MT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) y[nt][mt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    const floatx4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    auto turn_x = [&](uint4 (&x)[MT][PLANES]) { // PLANES == 2: the operands already
        if constexpr (PLANES == 1) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) *(uint4 *)(s_x + 16 * STRIDE * mt + put) = x[mt][0];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) x[mt][0] = *(const uint4 *)(s_x + 16 * STRIDE * mt + get);
        }
    };
    auto multiply = [&](uint32_t b, const uint2 (&w)[NT], const uint4 (&x)[MT][PLANES]) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const bf16x8 wb = q8_codes_to_bf16_perm(w[nt]);
            const float sc = f16_bits_to_f32(s_sc[s_row[nt] + b]);
            floatx4 acc[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(x[mt][0]), wb, zero4, 0, 0, 0);
            if constexpr (PLANES == 2) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(x[mt][1]), wb, acc[mt], 0, 0, 0);
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
                for (int i = 0; i < 4; ++i) y[nt][mt][i] = __builtin_fmaf(sc, acc[mt][i], y[nt][mt][i]);
            }
        }
    };

    uint4 w_next[NT], xa[MT][PLANES], xb[MT][PLANES];
    // whole pairs; a block left over is the last wavefront's, a turn of its own after them (the runs of lng_q8_few*: the same
    // sums in the same order)
    const uint32_t full = blocks / 2u, pairs = (blocks + 1u) / 2u;
    const uint32_t from = wave * pairs / NW, to = wave == NW - 1u ? full : (wave + 1u) * pairs / NW;
    if (from < to) {
        load_w(from, w_next);
        load_x(2u * from, xa);
    }
    // the tile's scales are one contiguous run; an odd one at its end, or a run off a 4-byte boundary, goes halfword by halfword
    const uint32_t count = rows_here * blocks;
    if (((uintptr_t)sc_src & 3u) == 0) {
        for (uint32_t i = threadIdx.x; i < count / 2u; i += 64u * NW) ((uint32_t *)s_sc)[i] = ((const uint32_t *)sc_src)[i];
        if ((count & 1u) && threadIdx.x == 0) s_sc[count - 1u] = sc_src[count - 1u];
    } else {
        for (uint32_t i = threadIdx.x; i < count; i += 64u * NW) s_sc[i] = sc_src[i];
    }
    __syncthreads();
    // The fences keep the loads where they are written, a block ahead of their use: left alone, the compiler moves them
    // down to the products that need them and every one is waited for in full.
    for (uint32_t pair = from; pair < to; ++pair) {
        uint2 w0[NT], w1[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const auto s0 = __builtin_amdgcn_permlane32_swap(w_next[nt].x, w_next[nt].z, false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(w_next[nt].y, w_next[nt].w, false, false);
            w0[nt] = make_uint2(s0[0], s1[0]);
            w1[nt] = make_uint2(s0[1], s1[1]);
        }
        const uint32_t next = pair + 1u < to ? pair + 1u : pair; // the last turn loads its own again
        load_w(next, w_next);
        load_x(2u * pair + 1u, xb);
        __builtin_amdgcn_sched_barrier(0);
        turn_x(xa);
        multiply(2u * pair, w0, xa);
        load_x(2u * next, xa);
        __builtin_amdgcn_sched_barrier(0);
        turn_x(xb);
        multiply(2u * pair + 1u, w1, xb);
    }
    if ((blocks & 1u) && wave == NW - 1u) {
        load_w(full, w_next);
        load_x(2u * full, xa);
        uint2 w0[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) { // the upper lanes hold the block again: their halves of it are what the swap takes
            const auto s0 = __builtin_amdgcn_permlane32_swap(w_next[nt].x, w_next[nt].z, false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(w_next[nt].y, w_next[nt].w, false, false);
            w0[nt] = make_uint2(s0[0], s1[0]);
        }
        turn_x(xa);
        multiply(2u * full, w0, xa);
    }
    __syncthreads(); // the scales and the turning buffers are dead
    float4 *s_red = (float4 *)s_mem; // [NW][NT * MT][64]
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            s_red[(wave * NT * MT + nt * MT + mt) * 64u + lane] = make_float4(y[nt][mt][0], y[nt][mt][1], y[nt][mt][2], y[nt][mt][3]);
        }
    }
    constexpr int MINE = (NT * MT + NW - 1) / NW; // of the tile's 16 x 16 parts
    float bias[MINE] = {}, held[MINE][4] = {};    // what is added, asked for while the partial results meet
#pragma unroll
    for (int m = 0; m < MINE; ++m) {
        const uint32_t at = wave + NW * m, row = 16u * (at / MT) + j, first = p0 + 16u * (at % MT) + 4u * kg;
        if (at < NT * MT && row < rows_here) {
            if (a.bias) bias[m] = a.bias[r0 + row];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (first + i < a.n && a.accumulate) held[m][i] = a.y[(uint64_t)(first + i) * a.y_stride + r0 + row];
                if (first + i < a.n && a.residual) held[m][i] = a.residual[(uint64_t)(first + i) * a.rows + r0 + row]; // never both
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MINE; ++m) {
        const uint32_t at = wave + NW * m;
        if (at >= NT * MT) break;
        float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float4 part = s_red[(w * NT * MT + at) * 64u + lane];
            sum[0] += part.x, sum[1] += part.y, sum[2] += part.z, sum[3] += part.w;
        }
        const uint32_t row = 16u * (at / MT) + j;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t p = p0 + 16u * (at % MT) + 4u * kg + i; // accumulator row = position, column = matrix row
            if (p < a.n && row < rows_here) {
                if (a.bias) sum[i] = sum[i] + bias[m];
                if (a.accumulate) sum[i] = held[m][i] + sum[i]; // the residual: h + ((W x) + bias), rounded as the separate dispatches round it
                a.y[(uint64_t)p * a.y_stride + r0 + row] = sum[i];
                if (a.residual) a.residual[(uint64_t)p * a.rows + r0 + row] = held[m][i] + sum[i];
            }
        }
    }
}

// Workgroup ids go round the eight XCDs, each with an L2 of its own: XCD k takes the row tiles k, k + 8, .. with all
// their position tiles one after another, so a row tile's codes come from memory once. ids without a tile leave.
template <int NT, int MT, int PLANES, int NW> __device__ __forceinline__ void q8_mid(lng_k_q8 a) {
    extern __shared__ __attribute__((aligned(16))) char s_mem[]; // as many bytes as q8_record_mid works out
    const uint32_t pos_tiles = (a.n + 16u * MT - 1u) / (16u * MT);
    const uint32_t seq = blockIdx.x >> 3;
    uint32_t row_tile = (seq / pos_tiles) * 8u + (blockIdx.x & 7u);
    const uint32_t pos_tile = seq % pos_tiles;
    if (row_tile >= a.tiles) return;
#pragma unroll
    for (int i = 0; i < LNG_Q8_MORE; ++i) { // several matrices: which one the tile belongs to (uniform: scalar selects)
        if ((uint32_t)i < a.n_more && row_tile >= a.more[i].first_tile) {
            a.codes = a.more[i].codes;
            a.scales = a.more[i].scales;
            a.y = a.more[i].y;
            a.rows = a.more[i].rows;
            a.y_stride = a.more[i].y_stride;
        }
    }
    uint32_t first = 0;
#pragma unroll
    for (int i = 0; i < LNG_Q8_MORE; ++i) {
        if ((uint32_t)i < a.n_more && row_tile >= a.more[i].first_tile) first = a.more[i].first_tile;
    }
    q8_mid_body<NT, MT, PLANES, NW>(a, row_tile - first, pos_tile, s_mem);
}

#define Q8_MID(name, nt, mt, planes, nw, per_simd) \
    extern "C" __global__ __launch_bounds__(64 * nw, per_simd) void name(lng_k_q8 a) { q8_mid<nt, mt, planes, nw>(a); }
Q8_MID(lng_q8_mid_r32p32, 2, 2, 2, 8, 4)
Q8_MID(lng_q8_mid_r64p64, 4, 4, 2, 4, 2)
Q8_MID(lng_q8_mid_bf16_r16p32, 1, 2, 1, 8, 4)
Q8_MID(lng_q8_mid_bf16_r32p64, 2, 4, 1, 4, 4)
Q8_MID(lng_q8_mid_bf16_r64p64, 4, 4, 1, 4, 2)
