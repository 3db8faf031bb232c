// The host library on the null device (loadngo_amd/csrc/null_device), under AddressSanitizer and
// UndefinedBehaviorSanitizer: what lng_hip.cpp decides before anything reaches a GPU.
//
//  - refusals: the reference's own rejected shapes (metal-compute/tests/attention_grouped.rs:262-279), slices of the
//    wrong length, outside their buffer or off their element size (apple.rs:860-887), outputs in resident memory or
//    over an input (apple.rs:889-906), buffers that belong to a batch in flight, and the refusals of copy_rows,
//    prepare_attention and the Q8_0 products; a refused call records nothing.
//  - the kernels that Q8_0 products are recorded as, and the sequences that a commit makes one kernel of: which do, with
//    which arguments, and which only look alike.
//  - the development switches (environment at open, lng_hip_debug_set afterwards) and lng_hip_checksum: refusals and
//    what is recorded.
//  - ownership: batches hand their buffers back; close with buffers alive; the last buffer freed on one thread while
//    the handle is closed on another.
//  - allocation failures while recording: reported, nothing recorded, nothing leaked.
//  - a fuzz of the decode planner: random tables of rows through lng_hip_attention_decode_batched and random
//    row-by-row calls; for every recorded dispatch the grid is the sum of the rows' live workgroups, every
//    (row, kv head, chunk) is taken by exactly one workgroup (the kernel's own search restated below), every chunk
//    has positions, the partials and arrival counters it names lie inside the scratch that was allocated, and the
//    merge that must follow does.
//
// Usage: null_device [fuzz dispatches, default 100000]. Exit status 0 = everything held.
#include <hip/hip_runtime_api.h> // the null device's

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <string>
#include <thread>
#include <tuple>
#include <vector>

#include "../../include/lng_hip.h"
#include "../../loadngo_amd/csrc/lng_kernel_args.h"

static int g_failures = 0;
#define CHECK(cond)                                                                      \
    do {                                                                                 \
        if (!(cond)) {                                                                   \
            fprintf(stderr, "%s:%d: CHECK failed: %s (last error: %s)\n", __FILE__, __LINE__, #cond, lng_hip_last_error()); \
            if (++g_failures > 20) exit(1);                                              \
        }                                                                                \
    } while (0)

static bool refused(int rc, const char *needle) {
    if (rc != LNG_ERR_DISPATCH) return false;
    return strstr(lng_hip_last_error(), needle) != nullptr;
}

static lng_grouped_shape shape(uint64_t t, uint64_t start, uint64_t heads, uint64_t kv_heads, uint64_t dim, uint64_t window,
                               uint64_t slots, float scale = 1.0f) {
    return lng_grouped_shape{t, start, heads, kv_heads, dim, window, slots, scale};
}

struct Fixture {
    lng_gpu *gpu = nullptr;
    std::vector<lng_buffer *> bufs;
    lng_batch *batch = nullptr;
    Fixture(size_t n, size_t bytes) {
        CHECK(lng_hip_open(0, &gpu) == LNG_OK);
        for (size_t i = 0; i < n; ++i) {
            lng_buffer *b = nullptr;
            CHECK(lng_hip_buffer(gpu, bytes, &b) == LNG_OK);
            bufs.push_back(b);
        }
        CHECK(lng_hip_batch(gpu, bufs.data(), bufs.size(), &batch) == LNG_OK);
    }
    void rebatch() {
        lng_hip_batch_drop(batch);
        CHECK(lng_hip_batch(gpu, bufs.data(), bufs.size(), &batch) == LNG_OK);
    }
    ~Fixture() {
        if (batch) lng_hip_batch_drop(batch);
        for (lng_buffer *b : bufs) CHECK(lng_hip_buffer_free(b) == LNG_OK);
        lng_hip_close(gpu);
    }
};

static void refusals() {
    const uint64_t MB = 1u << 20;
    Fixture f(5, MB);
    lng_batch *b = f.batch;
    auto whole = [&](uint64_t i) { return lng_slice{i, 0, MB}; };
    // attention_grouped.rs:262-279
    const lng_grouped_shape rejected[] = {shape(1, 0, 6, 4, 64, 8, 8), shape(1, 0, 4, 4, 48, 8, 8), shape(1, 0, 4, 4, 544, 8, 8),
                                          shape(4, 100, 4, 4, 64, 8, 10), shape(0, 0, 4, 4, 64, 8, 8)};
    for (const lng_grouped_shape &s : rejected) {
        CHECK(refused(lng_hip_attention_grouped(b, whole(0), whole(1), whole(2), whole(3), nullptr, &s, LNG_F32), "unsupported"));
        CHECK(lng_hip_check_grouped(&s, 0) == LNG_ERR_DISPATCH);
    }
    // tiled: the ring must be a multiple of 32 rows (apple.rs:1356-1385)
    {
        const lng_grouped_shape s = shape(40, 97, 4, 1, 64, 7, 50);
        CHECK(lng_hip_check_grouped(&s, 1) == LNG_ERR_DISPATCH);
        const lng_grouped_shape ok = shape(40, 97, 4, 1, 64, 7, 64);
        CHECK(lng_hip_check_grouped(&ok, 1) == LNG_OK);
    }
    // counts past u32
    {
        const lng_grouped_shape s = shape(1, 1ull << 33, 4, 4, 64, 8, 8);
        CHECK(lng_hip_check_grouped(&s, 0) == LNG_ERR_DISPATCH);
    }
    CHECK(lng_hip_batch_dispatches(b) == 0 && lng_null_launch_count() == 0);

    // a good call, then every way its slices can be wrong (apple.rs:860-906)
    const lng_grouped_shape s = shape(2, 5, 8, 2, 64, LNG_WINDOW_FULL, 16);
    const uint64_t qn = 2 * 8 * 64 * 4, kn = 7 * 2 * 64 * 4;
    const lng_slice q{0, 0, qn}, k{1, 0, kn}, v{2, 0, kn}, o{3, 0, qn}, sk{4, 0, 8 * 4};
    CHECK(lng_hip_attention_grouped(b, q, k, v, o, &sk, &s, LNG_F32) == LNG_OK);
    CHECK(lng_hip_batch_dispatches(b) == 1);
    lng_slice bad = q;
    bad.len -= 4;
    CHECK(refused(lng_hip_attention_grouped(b, bad, k, v, o, &sk, &s, LNG_F32), "the shape needs"));
    bad = k;
    bad.offset = MB - kn + 4;
    CHECK(refused(lng_hip_attention_grouped(b, q, bad, v, o, &sk, &s, LNG_F32), "outside"));
    bad = v;
    bad.offset = 2;
    CHECK(refused(lng_hip_attention_grouped(b, q, k, bad, o, &sk, &s, LNG_F32), "not a multiple"));
    bad = o;
    bad.buffer = 9;
    CHECK(refused(lng_hip_attention_grouped(b, q, k, v, bad, &sk, &s, LNG_F32), "no buffer"));
    bad = lng_slice{0, qn / 2, qn}; // output over the query
    CHECK(refused(lng_hip_attention_grouped(b, q, k, v, bad, &sk, &s, LNG_F32), "overlaps"));
    bad = sk;
    bad.len = 4;
    CHECK(refused(lng_hip_attention_grouped(b, q, k, v, o, &bad, &s, LNG_F32), "the shape needs"));
    CHECK(refused(lng_hip_attention_grouped(b, q, k, v, o, &sk, &s, 7), "unknown element type"));
    CHECK(refused(lng_hip_attention_grouped(b, q, k, v, o, &sk, nullptr, LNG_F32), "no shape"));
    CHECK(lng_hip_batch_dispatches(b) == 1);

    // resident memory is never an output (apple.rs:896-900)
    std::vector<char> bytes(qn, 1);
    lng_buffer *res = nullptr;
    CHECK(lng_hip_resident(f.gpu, bytes.data(), bytes.size(), &res) == LNG_OK);
    lng_slice rs{};
    CHECK(lng_hip_batch_attach(b, res, &rs) == LNG_OK && rs.buffer == 5 && rs.len == qn);
    CHECK(refused(lng_hip_attention_grouped(b, q, k, v, rs, &sk, &s, LNG_F32), "read-only resident"));
    CHECK(lng_hip_attention_grouped(b, rs, k, v, o, &sk, &s, LNG_F32) == LNG_OK); // ... but an input
    CHECK(refused(lng_hip_batch_attach(b, f.bufs[0], &rs), "not a resident"));
    CHECK(refused(lng_hip_upload(res, 0, bytes.data(), 4), "read-only"));
    CHECK(refused(lng_hip_buffer_free(res), "belongs to a batch"));

    // copy_rows (apple.rs:1769-1781)
    CHECK(refused(lng_hip_copy_rows(b, whole(0), 64, LNG_F32, whole(1), 64, LNG_F32, 0, 64), "unsupported copy"));
    CHECK(refused(lng_hip_copy_rows(b, whole(0), 32, LNG_F32, whole(1), 64, LNG_F32, 4, 64), "unsupported copy"));
    CHECK(refused(lng_hip_copy_rows(b, lng_slice{0, 0, 4 * 64 * 4}, 64, LNG_F32, lng_slice{0, 64, 4 * 64 * 4}, 64, LNG_F32, 4, 64), "overlaps"));
    CHECK(lng_hip_copy_rows(b, lng_slice{0, 0, (3 * 80 + 64) * 4}, 80, LNG_F32, lng_slice{1, 0, (3 * 64 + 64) * 2}, 64, LNG_BF16, 4, 64) == LNG_OK);
    // rmsnorm / add_rows / rotate_halves (apple.rs:1740-1744, 1893-1897, 1936-1940)
    CHECK(refused(lng_hip_rmsnorm_rows(b, whole(0), lng_slice{1, 0, 64 * 4}, 4, 64, 32, 1e-5f), "unsupported rows"));
    CHECK(refused(lng_hip_add_rows(b, whole(0), whole(1), 8, 4, 64), "unsupported add"));
    CHECK(refused(lng_hip_rotate_halves(b, whole(0), whole(1), 4, 8, 64, 65), "unsupported"));
    // Q8_0 products: columns in whole blocks, codes and x on 16-byte boundaries
    CHECK(lng_hip_gemv_q8_0(b, lng_slice{0, 0, 64 * 96}, lng_slice{1, 0, 64 * 3 * 2}, lng_slice{2, 0, 96 * 4}, lng_slice{3, 0, 64 * 4}, 64, 96) == LNG_OK);
    CHECK(lng_hip_gemv_q8_0(b, lng_slice{0, 0, 64 * 90}, lng_slice{1, 0, 64 * 3 * 2}, lng_slice{2, 0, 90 * 4}, lng_slice{3, 0, 64 * 4}, 64, 90) == LNG_ERR_DISPATCH);
    CHECK(lng_hip_gemv_q8_0(b, lng_slice{0, 4, 64 * 96}, lng_slice{1, 0, 64 * 3 * 2}, lng_slice{2, 0, 96 * 4}, lng_slice{3, 0, 64 * 4}, 64, 96) == LNG_ERR_DISPATCH);
    CHECK(lng_hip_gemm_q8_0_tiled(b, lng_slice{0, 0, 64 * 96}, lng_slice{1, 0, 64 * 3 * 2}, lng_slice{2, 0, 33 * 96 * 4}, lng_slice{3, 0, 33 * 64 * 4}, 64, 96, 33, 96, 64) == LNG_ERR_DISPATCH);
    // the fused pre-attention step: two new rows on one cache row, outputs over one another
    {
        lng_prepare_buffers pb{0, 1, 2, 4, 3, 3, 3, nullptr, nullptr, nullptr};
        lng_prepare_item it{};
        it.n = 4, it.start = 0, it.slots = 2;
        CHECK(refused(lng_hip_prepare_attention(b, &pb, &it, 1, 8, 2, 64, 64, LNG_BF16), "unsupported preparation"));
        it.slots = 8; // q_out, k and v caches all at offset 0 of buffer 3
        CHECK(refused(lng_hip_prepare_attention(b, &pb, &it, 1, 8, 2, 64, 64, LNG_BF16), "overlap"));
    }
    // decode items: outputs of two items over one another
    {
        lng_decode_item items[2] = {};
        for (lng_decode_item &it : items) it = lng_decode_item{0, 0, 0, 0, LNG_NO_SINKS, 3, LNG_WINDOW_FULL, 4};
        items[1].q_offset = 8 * 64 * 2;
        CHECK(refused(lng_hip_attention_decode_batched(b, 0, 1, 2, 3, 4, items, 2, 8, 2, 64, 0.125f, LNG_BF16), "overlap"));
        items[1].out_offset = 8 * 64 * 2;
        CHECK(lng_hip_attention_decode_batched(b, 0, 1, 2, 3, 4, items, 2, 8, 2, 64, 0.125f, LNG_BF16) == LNG_OK);
        items[1].start = 9; // a row the cache cannot hold
        CHECK(lng_hip_attention_decode_batched(b, 0, 1, 2, 3, 4, items, 2, 8, 2, 64, 0.125f, LNG_BF16) == LNG_ERR_DISPATCH);
    }

    // ownership: while the batch is alive its buffers are its own (apple.rs:365-389)
    char word[4] = {0};
    CHECK(refused(lng_hip_upload(f.bufs[0], 0, word, 4), "belongs to a batch"));
    CHECK(refused(lng_hip_download(f.bufs[0], 0, word, 4), "belongs to a batch"));
    CHECK(refused(lng_hip_buffer_free(f.bufs[0]), "belongs to a batch"));
    lng_batch *second = nullptr;
    CHECK(refused(lng_hip_batch(f.gpu, f.bufs.data(), 1, &second), "belongs to a batch") && second == nullptr);
    lng_buffer *twice[2] = {res, res};
    CHECK(lng_hip_batch(f.gpu, twice, 2, &second) == LNG_ERR_DISPATCH); // a resident is attached, not owned
    const size_t recorded = lng_hip_batch_dispatches(b);
    CHECK(lng_null_launch_count() == 0); // nothing runs before commit (apple.rs:553-561)
    double seconds = -1.0;
    CHECK(refused(lng_hip_batch_wait(b, &seconds), "not committed"));
    CHECK(lng_hip_batch_commit(b, nullptr, nullptr) == LNG_OK);
    CHECK(lng_null_launch_count() >= recorded);
    CHECK(refused(lng_hip_attention_grouped(b, q, k, v, o, &sk, &s, LNG_F32), "already committed"));
    CHECK(lng_hip_batch_wait(b, &seconds) == LNG_OK && seconds >= 0.0);
    CHECK(lng_hip_upload(f.bufs[0], 0, word, 4) == LNG_OK); // the buffers are the caller's again
    CHECK(lng_hip_upload(f.bufs[0], MB - 2, word, 4) == LNG_ERR_DISPATCH);
    f.rebatch();
    CHECK(lng_hip_buffer_free(res) == LNG_OK);
    lng_null_clear();
}

static std::vector<std::string> launched() { // the kernels launched since the last clear, in order
    std::vector<std::string> names;
    for (size_t i = 0; i < lng_null_launch_count(); ++i) {
        const char *name = nullptr;
        CHECK(lng_null_launch(i, &name, nullptr, nullptr, nullptr, nullptr) == 0);
        names.push_back(name);
    }
    return names;
}

// Which kernels Q8_0 products run as.
// 32 positions or more: lng_q8_mid* where the tiles of lng_q8_tiled would leave units idle, lng_q8_tiled where
// they fill the device, whichever number of positions; a matrix takes the same kernel alone and among others.
static void products_and_their_kernels() {
    Fixture f(4, 66ull << 20);
    const uint64_t cols = 512;
    auto run = [&]() {
        CHECK(lng_hip_batch_commit(f.batch, nullptr, nullptr) == LNG_OK);
        CHECK(lng_hip_batch_wait(f.batch, nullptr) == LNG_OK);
        const std::vector<std::string> names = launched();
        lng_null_clear();
        f.rebatch();
        return names;
    };
    auto product = [&](uint64_t rows, uint64_t n, bool bf16) {
        const lng_slice codes{0, 0, rows * cols}, scales{1, 0, rows * cols / 16}, x{2, 0, n * cols * (bf16 ? 2u : 4u)}, y{3, 0, n * rows * 4};
        CHECK((bf16 ? lng_hip_gemm_q8_0_bf16 : lng_hip_gemm_q8_0)(f.batch, codes, scales, x, y, rows, cols, n, cols, rows) == LNG_OK);
        return run().back();
    };
    const struct { uint64_t rows, n; bool bf16; const char *kernel; } wanted[] = {
        {2880, 32, false, "lng_q8_mid_r32p32"}, {2880, 129, false, "lng_q8_mid_r64p64"}, {2880, 512, false, "lng_q8_mid_r64p64"}, {2880, 1281, false, "lng_q8_tiled"},
        {65536, 128, false, "lng_q8_tiled"}, {32768, 512, false, "lng_q8_tiled"}, {16384, 512, false, "lng_q8_tiled"}, {16384, 32, false, "lng_q8_mid_r32p32"},
        {65536, 31, false, "lng_q8_mid_r32p32"},
        {2880, 32, true, "lng_q8_mid_bf16_r16p32"}, {2880, 77, true, "lng_q8_mid_bf16_r32p64"}, {2880, 512, true, "lng_q8_mid_bf16_r64p64"}, {2880, 1281, true, "lng_q8_tiled_bf16"},
        {65536, 128, true, "lng_q8_tiled_bf16"}, {16384, 512, true, "lng_q8_tiled_bf16"}, {65536, 17, true, "lng_q8_mid_bf16_r16p32"}};
    for (const auto &w : wanted) {
        const std::string kernel = product(w.rows, w.n, w.bf16);
        if (kernel != w.kernel) fprintf(stderr, "%llu rows, %llu positions, bf16 %d: %s\n", (unsigned long long)w.rows, (unsigned long long)w.n, w.bf16, kernel.c_str());
        CHECK(kernel == w.kernel);
    }
    // several matrices: those of many rows after the dispatch that the others share, each with the kernel it takes alone
    const uint64_t n = 128, rows[3] = {512, 62464, 2560}, at[3] = {0, 512, 62976};
    lng_q8_matrix m[3];
    for (int i = 0; i < 3; ++i) m[i] = {{0, at[i] * cols, rows[i] * cols}, {1, at[i] * cols / 16, rows[i] * cols / 16}, {3, at[i] * n * 4, rows[i] * n * 4}, rows[i]};
    CHECK(lng_hip_gemm_q8_0_many(f.batch, m, 3, lng_slice{2, 0, n * cols * 4}, cols, n, cols) == LNG_OK);
    CHECK(lng_hip_batch_dispatches(f.batch) == 3);
    const std::vector<std::string> names = run();
    CHECK((names == std::vector<std::string>{"lng_q8_frag_x", "lng_q8_mid_r32p32", "lng_q8_split_x", "lng_q8_tiled"}));
    // one position: past as many tiles of 16 rows as the device holds workgroups, each workgroup takes several
    const struct { uint64_t rows, cols; bool bf16; const char *kernel; uint32_t grid, tile, tiles; } ones[] = {
        {8192, 96, false, "lng_q8_one", 512, 16, 512}, {8193, 96, false, "lng_q8_tall", 512, 16, 513}, {65536, 96, true, "lng_q8_tall_bf16", 512, 16, 4096},
        {2880, 2880, true, "lng_q8_one_bf16", 240, 12, 240}, {4096, 12288, false, "lng_q8_one", 256, 16, 256}, {4097, 12288, false, "lng_q8_tall", 256, 16, 257}};
    for (const auto &w : ones) {
        const lng_slice x{2, 0, w.cols * (w.bf16 ? 2u : 4u)}, y{3, 0, w.rows * 4};
        CHECK((w.bf16 ? lng_hip_gemm_q8_0_bf16 : lng_hip_gemm_q8_0)(f.batch, lng_slice{0, 0, w.rows * w.cols}, lng_slice{1, 0, w.rows * w.cols / 16}, x, y, w.rows, w.cols, 1, w.cols, w.rows) == LNG_OK);
        CHECK(lng_hip_batch_commit(f.batch, nullptr, nullptr) == LNG_OK && lng_hip_batch_wait(f.batch, nullptr) == LNG_OK);
        const std::vector<std::string> names = launched();
        const char *name = nullptr;
        unsigned grid[3], block[3];
        const void *args = nullptr;
        size_t size = 0;
        CHECK(names == std::vector<std::string>{w.kernel} && lng_null_launch(0, &name, grid, block, &args, &size) == 0 && size == sizeof(lng_k_q8));
        const lng_k_q8 *a = (const lng_k_q8 *)args;
        if (grid[0] != w.grid || a->one_rows != w.tile || a->tiles != w.tiles) fprintf(stderr, "%llu x %llu: %u workgroups, %u tiles of %u\n", (unsigned long long)w.rows, (unsigned long long)w.cols, grid[0], a->tiles, a->one_rows);
        CHECK(grid[0] == w.grid && a->one_rows == w.tile && a->tiles == w.tiles && block[0] == 512);
        lng_null_clear();
        f.rebatch();
    }
    // 2 to 31 positions: f32 ones are split by the product itself where that is less than a dispatch before it
    typedef std::vector<std::string> Names;
    auto few = [&](uint64_t rows, uint64_t cols, uint64_t n, bool normed) {
        const lng_slice x{2, 0, n * cols * 4}, norm{2, x.len, cols * 4};
        const lng_q8_matrix m{{0, 0, rows * cols}, {1, 0, rows * cols / 16}, {3, 0, n * rows * 4}, rows};
        if (normed) CHECK(lng_hip_gemm_q8_0_many_normed(f.batch, &m, 1, x, norm, 1e-5f, cols, n, cols) == LNG_OK);
        else CHECK(lng_hip_gemm_q8_0(f.batch, m.codes, m.scales, x, m.y, rows, cols, n, cols, rows) == LNG_OK);
        return run();
    };
    for (const bool normed : {false, true}) {
        CHECK(few(2880, 512, 2, normed) == Names{"lng_q8_few_f32"});
        CHECK(few(4096, 512, 16, normed) == Names{"lng_q8_few_f32"});
        CHECK((few(2880, 2880, 16, normed) == Names{"lng_q8_norm_frag", "lng_q8_few"}));
        CHECK(few(2048, 512, 31, normed) == Names{"lng_q8_few_f32"});
        CHECK((few(2880, 2880, 31, normed) == Names{"lng_q8_norm_frag", "lng_q8_few"}));
        CHECK((few(4096, 2880, 31, normed) == Names{"lng_q8_norm_frag", "lng_q8_mid_r32p32"}));
        // 2 to 16 positions of 2,048 to 4,096 columns and more rows than a workgroup of 16 a unit takes, up to 32
        const Names planes{"lng_q8_norm_frag", "lng_q8_few"}, split{"lng_q8_few_split"};
        CHECK(few(4096, 2880, 16, normed) == planes && few(4097, 2880, 16, normed) == split && few(8192, 2880, 16, normed) == split && few(8193, 2880, 16, normed) == planes);
        CHECK(few(5120, 2016, 16, normed) == planes && few(5120, 2048, 16, normed) == split && few(5120, 4096, 16, normed) == split && few(5120, 4128, 16, normed) == planes);
        CHECK((few(5120, 2880, 17, normed) == Names{"lng_q8_norm_frag", "lng_q8_mid_r32p32"}) && few(5120, 2880, 2, normed) == split);
        CHECK(few(8192, 2880, 4, normed) == split && few(8192, 2880, 3, normed) == (normed ? split : Names{"lng_q8_few_f32"}));
    }
    lng_null_clear();
}

// One recorded launch by its name's beginning: its arguments, or NULL.
template <typename A> static bool launch_args(size_t i, const char *prefix, A *a, unsigned *grid0 = nullptr) {
    const char *name = nullptr;
    const void *args = nullptr;
    size_t size = 0;
    unsigned grid[3];
    if (lng_null_launch(i, &name, grid, nullptr, &args, &size) != 0 || strncmp(name, prefix, strlen(prefix)) != 0 || size < sizeof(A)) return false;
    memcpy(a, args, sizeof(A));
    if (grid0) *grid0 = grid[0];
    return true;
}

// Sequences of a block's dispatches that a commit makes one kernel of, and sequences that only look alike.
static void fused_sequences() {
    typedef std::vector<std::string> Names;
    Fixture f(9, 12 << 20);
    auto run = [&]() {
        CHECK(lng_hip_batch_commit(f.batch, nullptr, nullptr) == LNG_OK && lng_hip_batch_wait(f.batch, nullptr) == LNG_OK);
        return launched();
    };
    auto again = [&]() {
        lng_null_clear();
        f.rebatch();
    };

    // ---- copy + RMS norm + split before Q8_0 products ----
    {
        const uint64_t cols = 288, rows = 64;
        auto block = [&](uint64_t n, uint64_t copied, uint64_t normed, uint64_t x_stride) { // n positions of hidden rows (buffer 0), x in buffer 1
            const lng_slice h{0, 0, copied * cols * 4}, x{1, 0, ((copied - 1) * x_stride + cols) * 4}, v{1, 0, ((normed - 1) * x_stride + cols) * 4};
            CHECK(lng_hip_copy_rows(f.batch, h, cols, LNG_F32, x, x_stride, LNG_F32, copied, cols) == LNG_OK);
            CHECK(lng_hip_rmsnorm_rows(f.batch, v, lng_slice{2, 0, cols * 4}, normed, cols, x_stride, 1e-5f) == LNG_OK);
            CHECK(lng_hip_gemm_q8_0(f.batch, lng_slice{3, 0, rows * cols}, lng_slice{4, 0, rows * cols / 16}, lng_slice{1, 0, ((n - 1) * x_stride + cols) * 4},
                                    lng_slice{5, 0, n * rows * 4}, rows, cols, n, x_stride, rows) == LNG_OK);
        };
        lng_k_rmsnorm norm{};
        lng_k_q8 product{};
        unsigned grid = 0;
        block(77, 77, 77, cols);
        CHECK((run() == Names{"lng_rmsnorm_row8", "lng_q8_mid_r32p32"}));
        CHECK(launch_args(0, "lng_rmsnorm_row8", &norm, &grid) && launch_args(1, "lng_q8_mid", &product));
        CHECK(norm.planes == LNG_PLANES_OPERAND && norm.hi == product.x_hi && grid == 96 && norm.n_pad == 96 && norm.rows == 77 && norm.src != norm.v && norm.v == product.x);
        again();
        block(1300, 1300, 1300, cols);
        CHECK((run() == Names{"lng_rmsnorm_row8", "lng_q8_tiled"}));
        CHECK(launch_args(0, "lng_rmsnorm_row8", &norm, &grid) && launch_args(1, "lng_q8_tiled", &product));
        CHECK(norm.planes == LNG_PLANES_ROWS && norm.hi == product.x_hi && norm.lo == product.x_lo && grid == 1408 && norm.src != norm.v);
        again();
        block(77, 77, 76, cols); // the norm of fewer rows than are copied, the product of more than are normalised
        CHECK((run() == Names{"lng_copy_rows", "lng_rmsnorm_row8", "lng_q8_frag_x", "lng_q8_mid_r32p32"}));
        CHECK(launch_args(1, "lng_rmsnorm_row8", &norm) && norm.src == norm.v && norm.planes == LNG_PLANES_NONE);
        again();
        block(16, 16, 16, cols); // few positions: the copy is part of the norm, the product splits by itself
        CHECK((run() == Names{"lng_rmsnorm_row8", "lng_q8_few_f32"}));
        again();
        for (int how = 0; how < 2; ++how) { // timed, or switched off: every dispatch as its own kernels
            if (how) CHECK(lng_hip_debug_set(f.gpu, "LNG_NO_FUSING", "1") == LNG_OK);
            else CHECK(lng_hip_batch_set_timing(f.batch, 1) == LNG_OK);
            block(77, 77, 77, cols);
            CHECK((run() == Names{"lng_copy_rows", "lng_rmsnorm_row8", "lng_q8_frag_x", "lng_q8_mid_r32p32"}));
            again();
        }
        CHECK(lng_hip_debug_set(f.gpu, "LNG_NO_FUSING", nullptr) == LNG_OK);
        // a copy to other rows, a norm of other rows than the product's
        CHECK(lng_hip_copy_rows(f.batch, lng_slice{0, 0, 40 * cols * 4}, cols, LNG_F32, lng_slice{6, 0, 40 * cols * 4}, cols, LNG_F32, 40, cols) == LNG_OK);
        CHECK(lng_hip_rmsnorm_rows(f.batch, lng_slice{1, 0, 40 * cols * 4}, lng_slice{2, 0, cols * 4}, 40, cols, cols, 1e-5f) == LNG_OK);
        CHECK(lng_hip_gemm_q8_0(f.batch, lng_slice{3, 0, rows * cols}, lng_slice{4, 0, rows * cols / 16}, lng_slice{6, 0, 40 * cols * 4}, lng_slice{5, 0, 40 * rows * 4}, rows, cols, 40, cols, rows) == LNG_OK);
        CHECK((run() == Names{"lng_copy_rows", "lng_rmsnorm_row8", "lng_q8_frag_x", "lng_q8_mid_r32p32"}));
        again();
    }

    // ---- product + bias + residual ----
    const struct { uint64_t n; bool bf16; const char *kernel, *folded; } products[] = {
        {1, false, "lng_q8_one", "lng_q8_one"}, {7, false, "lng_q8_few_f32", "lng_q8_few_f32"}, {33, false, "lng_q8_mid_r32p32", "lng_q8_mid_r32p32"},
        {1290, false, "lng_q8_tiled", "lng_q8_tiled_add"}, {1, true, "lng_q8_one_bf16", "lng_q8_one_bf16"}, {16, true, "lng_q8_few_bf16", "lng_q8_few_bf16"},
        {129, true, "lng_q8_mid_bf16_r64p64", "lng_q8_mid_bf16_r64p64"}, {1290, true, "lng_q8_tiled_bf16", "lng_q8_tiled_bf16_add"}};
    for (const auto &w : products) {
        const uint64_t rows = 64, cols = 96, n = w.n, len = n * rows * 4;
        const lng_slice x{0, 0, n * cols * (w.bf16 ? 2u : 4u)}, codes{3, 0, rows * cols}, scales{4, 0, rows * cols / 16}, y{5, 0, len}, bias{2, 0, rows * 4}, h{6, 0, len};
        auto product = [&](uint64_t y_stride = 64) {
            const lng_slice out{5, 0, ((n - 1) * y_stride + rows) * 4};
            CHECK((w.bf16 ? lng_hip_gemm_q8_0_bf16 : lng_hip_gemm_q8_0)(f.batch, codes, scales, x, out, rows, cols, n, cols, y_stride) == LNG_OK);
        };
        auto add = [&](lng_slice dst, lng_slice src, uint64_t stride) { CHECK(lng_hip_add_rows(f.batch, dst, src, stride, n, rows) == LNG_OK); };
        auto last = [&](const char *kernel, size_t adds) { // the product (and what splits before it), then so many additions
            const Names names = run();
            const size_t at = names.size() - 1 - adds;
            CHECK(names.size() > adds && names[at] == kernel);
            for (size_t i = at + 1; i < names.size(); ++i) CHECK(names[i] == "lng_add_rows");
            return at;
        };
        lng_k_q8 a{};
        product(), add(y, bias, 0), add(h, y, rows);
        CHECK(launch_args(last(w.folded, 0), "lng_q8", &a) && a.bias && a.residual && a.residual != a.y && !a.accumulate);
        again();
        product(), add(h, y, rows), add(h, y, rows), add(y, bias, 0); // the residual, and what comes after it
        CHECK(launch_args(last(w.folded, 2), "lng_q8", &a) && !a.bias && a.residual);
        again();
        product(), add(y, bias, 0), add(y, bias, 0);
        CHECK(launch_args(last(w.folded, 1), "lng_q8", &a) && a.bias && !a.residual);
        again();
        if (n > 1) {
            product(68); // y with gaps
            CHECK(lng_hip_add_rows(f.batch, h, lng_slice{5, 0, ((n - 1) * 68 + rows) * 4}, 68, n, rows) == LNG_OK);
            CHECK(launch_args(last(w.kernel, 1), "lng_q8", &a) && !a.residual);
            again();
        }
        for (const lng_slice over : {lng_slice{0, 0, len}, lng_slice{3, 0, len}, lng_slice{4, 0, len}}) { // other workgroups still read what it is added to
            product(), add(over, y, rows);
            CHECK(launch_args(last(w.kernel, 1), "lng_q8", &a) && !a.residual);
            again();
        }
        product(), add(y, bias, 0), add(lng_slice{2, 0, len}, y, rows); // over the bias
        CHECK(launch_args(last(w.folded, 1), "lng_q8", &a) && a.bias && !a.residual);
        again();
    }

    for (const auto &w : {std::make_tuple(4u, 4112u, 2048u, "lng_q8_few_split"), std::make_tuple(1u, 9000u, 96u, "lng_q8_tall")}) {
        const uint64_t n = std::get<0>(w), rows = std::get<1>(w), cols = std::get<2>(w), len = n * rows * 4;
        const lng_slice y{5, 0, len}, bias{2, 0, rows * 4}, h{6, 0, len};
        CHECK(lng_hip_gemm_q8_0(f.batch, lng_slice{3, 0, rows * cols}, lng_slice{4, 0, rows * cols / 16}, lng_slice{0, 0, n * cols * 4}, y, rows, cols, n, cols, rows) == LNG_OK);
        CHECK(lng_hip_add_rows(f.batch, y, bias, 0, n, rows) == LNG_OK && lng_hip_add_rows(f.batch, h, y, rows, n, rows) == LNG_OK);
        lng_k_q8 a{};
        CHECK(run() == Names{std::get<3>(w)} && launch_args(0, "lng_q8", &a) && a.bias && a.residual && a.residual != a.y && !a.accumulate);
        again();
    }

    // ---- the q, k and v projections + the preparation of attention ----
    struct Case { uint64_t n, cols, rotary; bool normed, one_item; const char *kind; Names names; uint64_t heads = 6, kv = 2; };
    const Case cases[] = {
        {1, 96, 64, true, true, "", {"lng_q8_one_prepare"}},
        {4, 96, 64, true, false, "", {"lng_q8_few_f32_prepare"}},
        {16, 96, 64, false, true, "", {"lng_q8_few_f32_prepare"}},
        {4, 2880, 64, true, false, "", {"lng_q8_norm_frag", "lng_q8_few_prepare"}},
        {2, 2048, 64, true, false, "", {"lng_q8_few_split_prepare"}, 64, 8},
        {16, 2048, 64, false, true, "", {"lng_q8_few_split_prepare"}, 64, 8},
        {1, 96, 64, true, true, "", {"lng_q8_one_prepare"}, 112, 16}, // (more tiles than the device holds workgroups: one to each all the same)
        {17, 96, 64, true, false, "", {"lng_q8_few_f32", "lng_prepare"}},
        {4, 96, 32, true, false, "", {"lng_q8_few_f32", "lng_prepare"}},
        {4, 96, 64, true, false, "backwards", {"lng_q8_few_f32", "lng_prepare"}},
        {4, 96, 64, true, false, "swapped", {"lng_q8_few_f32", "lng_prepare"}},
        {4, 96, 64, true, false, "table over q", {"lng_q8_few_f32", "lng_prepare"}},
        {4, 96, 64, true, false, "queries over x", {"lng_q8_few_f32", "lng_prepare"}},
        {4, 96, 64, true, false, "biases over v", {"lng_q8_few_f32", "lng_prepare"}},
    };
    for (const Case &c : cases) {
        const uint64_t heads = c.heads, kv = c.kv, qw = heads * 64, kw = kv * 64, n = c.n, slots = 24;
        const std::string kind = c.kind;
        const uint64_t k_at = kind == "swapped" ? n * kw * 4 : 0, v_at = kind == "swapped" ? 0 : n * kw * 4;
        const lng_slice x{0, 0, n * c.cols * 4}, norm{2, 0, c.cols * 4};
        const uint64_t widths[3] = {qw, kw, kw};
        const lng_slice ys[3] = {{5, 0, n * qw * 4}, {6, k_at, n * kw * 4}, {6, v_at, n * kw * 4}};
        lng_q8_matrix m[3];
        uint64_t at = 0;
        for (int i = 0; i < 3; ++i) {
            m[i] = {{3, at * c.cols, widths[i] * c.cols}, {4, at * c.cols / 16, widths[i] * c.cols / 16}, ys[i], widths[i]};
            at += widths[i];
        }
        if (c.normed) CHECK(lng_hip_gemm_q8_0_many_normed(f.batch, m, 3, x, norm, 1e-5f, c.cols, n, c.cols) == LNG_OK);
        else CHECK(lng_hip_gemm_q8_0_many(f.batch, m, 3, x, c.cols, n, c.cols) == LNG_OK);
        const uint64_t biases_in = kind == "biases over v" ? 6 : 1, bias_at = kind == "biases over v" ? v_at : 0; // (read by the preparation only)
        const lng_slice qb{1, 0, qw * 4}, kb{biases_in, bias_at, kw * 4}, vb{1, 8192, kw * 4};
        const lng_prepare_buffers pb{5, 6, 6, (uint64_t)(kind == "table over q" ? 5 : 7), (uint64_t)(kind == "queries over x" ? 0 : 8), 7, 7, &qb, &kb, &vb};
        std::vector<lng_prepare_item> items;
        for (uint64_t i = 0; i < (c.one_item ? 1 : n); ++i) {
            const uint64_t j = kind == "backwards" ? n - 1 - i : i;
            lng_prepare_item it{};
            it.q_offset = j * qw * 4, it.k_offset = j * kw * 4, it.v_offset = n * kw * 4 + j * kw * 4, it.table_offset = (pb.table == 7 ? 3 << 20 : 0) + j * c.rotary * 4;
            it.q_out_offset = j * qw * 2, it.k_cache_offset = i * slots * kw * 2, it.v_cache_offset = (n + i) * slots * kw * 2;
            it.n = c.one_item ? n : 1, it.start = 5 + i, it.slots = slots;
            items.push_back(it);
        }
        CHECK(lng_hip_prepare_attention(f.batch, &pb, items.data(), items.size(), heads, kv, 64, c.rotary, LNG_BF16) == LNG_OK);
        const Names names = run();
        bool same = names.size() == c.names.size();
        for (size_t i = 0; same && i < names.size(); ++i) same = names[i].rfind(c.names[i], 0) == 0 && (c.names[i] == "lng_prepare" || names[i] == c.names[i]);
        if (!same) fprintf(stderr, "%llu positions, %llu columns, %llu rotated, %s: %zu launches, first %s\n", (unsigned long long)n, (unsigned long long)c.cols, (unsigned long long)c.rotary, c.kind, names.size(), names[0].c_str());
        CHECK(same);
        if (names.back().find("_prepare") != std::string::npos && names.back().rfind("lng_q8", 0) == 0) {
            lng_k_q8_prepare both{};
            CHECK(launch_args(names.size() - 1, "lng_q8", &both) && both.q8.n == n && both.q8.n_more == 2 && both.prepare.heads == heads && both.prepare.kv_heads == kv);
            unsigned grid = 0;
            CHECK(launch_args(names.size() - 1, "lng_q8", &both, &grid) && (!both.q8.one_rows || (grid == both.q8.tiles && both.q8.one_rows % 2 == 0)));
            CHECK((both.prepare.items == nullptr) == (items.size() == 1) && both.prepare.q_bias && both.prepare.k_bias && both.prepare.v_bias);
        }
        again();
    }
}

// The development switches (read from the environment once, at open; afterwards only lng_hip_debug_set) and the
// streaming read: refusals, and what the planner records under a switch.
static void switches_and_checksum() {
    const size_t MB = 1 << 20;
    setenv("LNG_PREFILL_SPLITS", "3", 1); // read at open ...
    Fixture f(5, MB);
    unsetenv("LNG_PREFILL_SPLITS"); // ... and never again
    lng_batch *b = f.batch;
    lng_null_clear();
    auto prefill_splits = [&]() { // a prompt pass of 64 rows over 1,024 cached positions: one query tile per kv head
        const lng_grouped_shape s = shape(64, 960, 8, 2, 64, LNG_WINDOW_FULL, 1024, 0.125f);
        const lng_slice q{0, 0, 64 * 8 * 64 * 2}, k{1, 0, 1024 * 2 * 64 * 2}, v{2, 0, 1024 * 2 * 64 * 2}, o{3, 0, 64 * 8 * 64 * 2};
        CHECK(lng_hip_attention_grouped_tiled(f.batch, q, k, v, o, nullptr, &s, LNG_BF16) == LNG_OK);
        CHECK(lng_hip_batch_commit(f.batch, nullptr, nullptr) == LNG_OK);
        CHECK(lng_hip_batch_wait(f.batch, nullptr) == LNG_OK);
        const char *name = nullptr;
        const void *args = nullptr;
        size_t args_size = 0;
        unsigned grid[3], block[3];
        CHECK(lng_null_launch_count() >= 1 && lng_null_launch(0, &name, grid, block, &args, &args_size) == 0);
        lng_k_prefill p{};
        CHECK(args_size == sizeof p);
        memcpy(&p, args, sizeof p);
        // (the kernel of a workgroup per pair of heads never splits: its grid has the pairs instead)
        const bool pairs = !strcmp(name, "lng_prefill_bf16_d64_pair");
        CHECK(grid[0] == p.q_tiles * p.kv_heads * (pairs ? (p.heads / p.kv_heads + 1) / 2 : p.splits));
        CHECK(!pairs || p.splits == 1);
        CHECK(p.splits == 1 || lng_null_launch_count() == 2);
        lng_null_clear();
        f.rebatch();
        return p.splits;
    };
    CHECK(prefill_splits() == 3); // the environment's value at open
    CHECK(lng_hip_debug_set(f.gpu, "LNG_PREFILL_SPLITS", "5") == LNG_OK);
    CHECK(prefill_splits() == 5);
    CHECK(lng_hip_debug_set(f.gpu, "LNG_PREFILL_SPLITS", nullptr) == LNG_OK);
    const uint32_t planned = prefill_splits(); // the planner's own: one workgroup per compute unit, four key tiles each at least
    CHECK(planned >= 1 && planned <= 4);
    // a prompt fed 512 rows at a time (64 heads over 8): 64 (query tile, kv head) pairs on 256 units go to the kernel of a
    // workgroup per pair of heads while a call walks few enough keys, and to split keys plus a merge beyond that
    {
        Fixture big(5, 40 * MB);
        auto chunk_call = [&](uint64_t start, const char *want_kernel, unsigned want_grid, size_t want_launches) {
            const lng_grouped_shape s = shape(512, start, 64, 8, 64, LNG_WINDOW_FULL, start + 512, 0.125f);
            const lng_slice q{0, 0, 512 * 64 * 64 * 2}, k{1, 0, (start + 512) * 8 * 64 * 2}, v{2, 0, (start + 512) * 8 * 64 * 2}, o{3, 0, 512 * 64 * 64 * 2};
            lng_null_clear();
            CHECK(lng_hip_attention_grouped_tiled(big.batch, q, k, v, o, nullptr, &s, LNG_BF16) == LNG_OK);
            CHECK(lng_hip_batch_commit(big.batch, nullptr, nullptr) == LNG_OK);
            CHECK(lng_hip_batch_wait(big.batch, nullptr) == LNG_OK);
            const char *name = nullptr;
            const void *args = nullptr;
            size_t args_size = 0;
            unsigned grid[3], block[3];
            CHECK(lng_null_launch_count() == want_launches && lng_null_launch(0, &name, grid, block, &args, &args_size) == 0);
            CHECK(!strcmp(name, want_kernel) && grid[0] == want_grid && block[0] == 512);
            big.rebatch();
        };
        const unsigned cus = 256; // the null device's
        chunk_call(3584, "lng_prefill_bf16_d64_pair", 8 * 8 * 4, 1);
        chunk_call(0, "lng_prefill_bf16_d64_pair", 8 * 8 * 4, 1);
        chunk_call(15872, "lng_prefill_bf16_d64", cus, 2);
        CHECK(lng_hip_debug_set(big.gpu, "LNG_PREFILL_PAIR", "0") == LNG_OK);
        chunk_call(3584, "lng_prefill_bf16_d64", cus, 2);
        CHECK(lng_hip_debug_set(big.gpu, "LNG_PREFILL_PAIR", "1") == LNG_OK);
        chunk_call(15872, "lng_prefill_bf16_d64_pair", 8 * 8 * 4, 1);
        CHECK(lng_hip_debug_set(big.gpu, "LNG_PREFILL_PAIR", nullptr) == LNG_OK);
        lng_null_clear();
    }
    // f32 passes: the keys are split where the time of the longest share and of every further round of workgroups is less
    {
        Fixture big(4, 24 * MB);
        auto splits = [&](uint64_t t, uint64_t start, uint64_t heads, uint64_t window, bool fails = false) {
            const uint64_t rows = (t + 31) / 32 * 32, kv = (start + t + 31) / 32 * 32;
            const lng_grouped_shape s = shape(t, start, heads, 8, 64, window, start + t, 0.125f);
            const lng_slice q{0, 0, rows * heads * 256}, k{1, 0, kv * 2048}, v{2, 0, kv * 2048}, o{3, 0, rows * heads * 256};
            lng_null_clear();
            lng_null_fail_malloc_after(fails ? 1 : 0);
            CHECK(lng_hip_attention_grouped_tiled(big.batch, q, k, v, o, nullptr, &s, LNG_F32) == LNG_OK);
            lng_null_fail_malloc_after(0);
            CHECK(lng_hip_batch_commit(big.batch, nullptr, nullptr) == LNG_OK && lng_hip_batch_wait(big.batch, nullptr) == LNG_OK);
            const void *args = nullptr;
            size_t args_size = 0;
            CHECK(lng_null_launch(0, nullptr, nullptr, nullptr, &args, &args_size) == 0 && args_size == sizeof(lng_k_prefill));
            lng_k_prefill p{};
            memcpy(&p, args, sizeof p);
            CHECK(lng_null_launch_count() == (p.splits > 1 ? 2 : 1));
            if (p.splits > 1) CHECK(lng_null_bytes_from(p.partial_o) >= t * heads * p.splits * 256);
            big.rebatch();
            return p.splits;
        };
        CHECK(splits(512, 0, 64, LNG_WINDOW_FULL, true) == 1); // no memory for partial rows
        CHECK(splits(512, 0, 64, LNG_WINDOW_FULL) == 4 && splits(256, 0, 64, LNG_WINDOW_FULL) == 4 && splits(64, 0, 64, LNG_WINDOW_FULL) == 1);
        CHECK(splits(48, 2000, 64, 128) > 1 && splits(256, 2000, 64, 128) == 4);
        CHECK(splits(673, 1000, 64, LNG_WINDOW_FULL) == 2 && splits(992, 4096, 64, LNG_WINDOW_FULL) == 2 && splits(1024, 0, 64, LNG_WINDOW_FULL) == 1);
        CHECK(splits(384, 0, 64, 128) == 1 && splits(450, 1000, 64, 128) == 1 && splits(512, 4096, 32, 128) == 1); // two tiles of keys: not worth a second round
        CHECK(splits(72, 0, 64, LNG_WINDOW_FULL) == 1 && splits(72, 0, 32, LNG_WINDOW_FULL) == 1);                 // nor the eight keys of a second
        CHECK(splits(300, 1000, 64, LNG_WINDOW_FULL) == 3 && splits(320, 1000, 32, LNG_WINDOW_FULL) == 3);         // one round of shares of seven against two of four
        lng_null_clear();
    }
    CHECK(refused(lng_hip_debug_set(f.gpu, "LNG_NO_SUCH_SWITCH", "1"), "no development switch"));
    CHECK(lng_hip_debug_set(f.gpu, "LNG_Q8_W16", "1") == LNG_OK && lng_hip_debug_set(f.gpu, "LNG_Q8_W16", nullptr) == LNG_OK); // of a kernel that is gone
    CHECK(refused(lng_hip_debug_set(f.gpu, nullptr, "1"), "no name"));
    CHECK(lng_hip_debug_set(nullptr, "LNG_PREFILL_SPLITS", "1") != LNG_OK);
    uint64_t n = 99;
    CHECK(lng_hip_debug_get(f.gpu, "LNG_COUNT_SECOND_PASSES", &n) == LNG_OK && n == 0);
    CHECK(refused(lng_hip_debug_get(f.gpu, "LNG_PREFILL_SPLITS", &n), "no development counter"));
    CHECK(lng_hip_debug_get(f.gpu, "LNG_COUNT_SECOND_PASSES", nullptr) != LNG_OK);

    // the streaming read: whole 16-byte words on a 16-byte boundary, 16 bytes out, not over its input
    b = f.batch;
    CHECK(refused(lng_hip_checksum(b, lng_slice{0, 0, 100}, lng_slice{1, 0, 16}), "16-byte words"));
    CHECK(refused(lng_hip_checksum(b, lng_slice{0, 0, 0}, lng_slice{1, 0, 16}), "16-byte words"));
    CHECK(refused(lng_hip_checksum(b, lng_slice{0, 8, 160}, lng_slice{1, 0, 16}), "not a multiple"));
    CHECK(refused(lng_hip_checksum(b, lng_slice{0, 0, 160}, lng_slice{1, 0, 32}), "the shape needs"));
    CHECK(refused(lng_hip_checksum(b, lng_slice{0, 0, 160}, lng_slice{1, 4, 16}), "not a multiple"));
    CHECK(refused(lng_hip_checksum(b, lng_slice{0, 0, 160}, lng_slice{0, 32, 16}), "overlaps"));
    CHECK(refused(lng_hip_checksum(b, lng_slice{0, MB - 16, 32}, lng_slice{1, 0, 16}), "outside"));
    CHECK(lng_hip_batch_dispatches(b) == 0);
    CHECK(lng_hip_checksum(b, lng_slice{0, 0, 160}, lng_slice{1, 0, 16}) == LNG_OK);       // ten words: one workgroup
    CHECK(lng_hip_checksum(b, lng_slice{0, 0, MB}, lng_slice{1, 16, 16}) == LNG_OK);        // 65,536 words: 256 workgroups
    CHECK(lng_hip_debug_set(f.gpu, "LNG_CHECKSUM_WGS", "1") == LNG_OK);
    CHECK(lng_hip_checksum(b, lng_slice{2, 0, MB}, lng_slice{1, 32, 16}) == LNG_OK);
    CHECK(lng_hip_batch_dispatches(b) == 3);
    CHECK(lng_hip_batch_commit(b, nullptr, nullptr) == LNG_OK);
    CHECK(lng_hip_batch_wait(b, nullptr) == LNG_OK);
    CHECK(lng_null_launch_count() == 6);
    for (size_t i = 0; i < 6; i += 2) {
        const char *name = nullptr, *fold = nullptr;
        const void *args = nullptr;
        size_t args_size = 0;
        unsigned grid[3], fgrid[3];
        CHECK(lng_null_launch(i, &name, grid, nullptr, &args, &args_size) == 0 && std::string(name) == "lng_checksum");
        CHECK(lng_null_launch(i + 1, &fold, fgrid, nullptr, nullptr, nullptr) == 0 && std::string(fold) == "lng_checksum_fold" && fgrid[0] == 1);
        lng_k_checksum a{};
        CHECK(args_size == sizeof a);
        memcpy(&a, args, sizeof a);
        CHECK(grid[0] == a.n_parts && a.n_parts >= 1 && a.n_parts <= (a.n16 + 255) / 256);
        CHECK(a.n16 == (i == 0 ? 10u : MB / 16));
        CHECK(lng_null_bytes_from(a.parts) >= (size_t)a.n_parts * 16); // a 16-byte word per workgroup, in the library's scratch
        CHECK(lng_null_bytes_from(a.src) >= a.n16 * 16 && lng_null_bytes_from(a.dst) >= 16);
        if (i == 0) CHECK(a.n_parts == 1);
        if (i == 4) { // one workgroup per compute unit instead of two
            lng_k_checksum two{};
            const void *args2 = nullptr;
            CHECK(lng_null_launch(2, nullptr, nullptr, nullptr, &args2, nullptr) == 0);
            memcpy(&two, args2, sizeof two);
            CHECK(two.n_parts == 256 ? a.n_parts <= 256 : a.n_parts * 2 == two.n_parts);
        }
    }
    lng_null_clear();
    f.rebatch();
}

static void on_done_count(const lng_completed *done, void *user) {
    if (done->status == LNG_OK) ++*(int *)user;
}

static void lifetimes() {
    // a committed batch with a callback, dropped from another thread than the completion thread
    {
        Fixture f(4, 1 << 16);
        const lng_grouped_shape s = shape(1, 3, 8, 2, 64, LNG_WINDOW_FULL, 8, 0.125f);
        const lng_slice q{0, 0, 8 * 64 * 2}, k{1, 0, 4 * 2 * 64 * 2}, v{2, 0, 4 * 2 * 64 * 2}, o{3, 0, 8 * 64 * 2};
        int done = 0;
        CHECK(lng_hip_attention_grouped(f.batch, q, k, v, o, nullptr, &s, LNG_BF16) == LNG_OK);
        CHECK(lng_hip_batch_commit(f.batch, on_done_count, &done) == LNG_OK);
        CHECK(lng_hip_batch_wait(f.batch, nullptr) == LNG_OK);
        CHECK(done == 1);
        f.rebatch();
    }
    // buffers outlive a closed device, whichever thread lets go last (the handle is one reference among them)
    for (int round = 0; round < 200; ++round) {
        lng_gpu *gpu = nullptr;
        CHECK(lng_hip_open(0, &gpu) == LNG_OK);
        lng_buffer *a = nullptr, *b = nullptr;
        CHECK(lng_hip_buffer(gpu, 256, &a) == LNG_OK && lng_hip_buffer(gpu, 256, &b) == LNG_OK);
        CHECK(lng_hip_buffer_free(a) == LNG_OK);
        std::thread closer([&] { lng_hip_close(gpu); });
        std::thread freer([&] { CHECK(lng_hip_buffer_free(b) == LNG_OK); });
        closer.join();
        freer.join();
    }
    CHECK(lng_null_live_allocations() == 0);
    lng_null_clear();
}

static void allocation_failures() {
    lng_gpu *gpu = nullptr;
    CHECK(lng_hip_open(0, &gpu) == LNG_OK);
    lng_buffer *buf = nullptr;
    lng_null_fail_malloc_after(1);
    CHECK(lng_hip_buffer(gpu, 1024, &buf) == LNG_ERR_ALLOC && buf == nullptr);
    CHECK(lng_hip_buffer(gpu, 0, &buf) == LNG_ERR_ALLOC); // Alloc(0), apple.rs:256-258
    // a decode that needs split-K scratch: the scratch allocation fails, the call is refused and records nothing
    const uint64_t ctx = 40000, row = 8 * 64 * 2;
    std::vector<lng_buffer *> bufs(4);
    const size_t sizes[4] = {64 * 64 * 2, ctx * row, ctx * row, 64 * 64 * 2};
    for (int i = 0; i < 4; ++i) CHECK(lng_hip_buffer(gpu, sizes[i], &bufs[i]) == LNG_OK);
    lng_batch *batch = nullptr;
    CHECK(lng_hip_batch(gpu, bufs.data(), 4, &batch) == LNG_OK);
    const lng_grouped_shape s = shape(1, ctx - 1, 64, 8, 64, LNG_WINDOW_FULL, ctx, 0.125f);
    const lng_slice q{0, 0, 64 * 64 * 2}, k{1, 0, ctx * row}, v{2, 0, ctx * row}, o{3, 0, 64 * 64 * 2};
    // the counters, the partial outputs, the (max, sum) pairs: each allocation fails once (what was allocated before
    // a failure stays with the device, so the second and third failures are the second allocation of their call)
    for (size_t nth : {1, 2, 2}) {
        lng_null_fail_malloc_after(nth);
        CHECK(lng_hip_attention_grouped(batch, q, k, v, o, nullptr, &s, LNG_BF16) == LNG_ERR_ALLOC);
        CHECK(lng_hip_batch_dispatches(batch) == 0);
        lng_null_fail_malloc_after(0);
    }
    CHECK(lng_hip_attention_grouped(batch, q, k, v, o, nullptr, &s, LNG_BF16) == LNG_OK);
    CHECK(lng_hip_batch_dispatches(batch) == 1);
    // f32 rows of 257 to 512 positions do without the partials when there is no memory for them, one row and a table; longer ones and
    // wider heads are refused
    const struct { uint64_t ctx, dim; bool whole; } rows_of[] = {{257, 64, true}, {300, 64, true}, {512, 64, true}, {513, 64, false}, {600, 128, false}};
    for (const auto &w : rows_of) {
        for (const bool table : {false, true}) {
            for (size_t nth = 1; nth <= 3; ++nth) { // the counters, the partial outputs, the (max, sum) pairs (after the table itself)
                Fixture f(4, 4 << 20);
                const uint64_t heads = 16, kv = 2, len = heads * w.dim * 4, cache = w.ctx * kv * w.dim * 4;
                const lng_grouped_shape one = shape(1, w.ctx - 1, heads, kv, w.dim, LNG_WINDOW_FULL, w.ctx, 0.125f);
                lng_decode_item items[2]{};
                for (int i = 0; i < 2; ++i) {
                    items[i].q_offset = items[i].out_offset = i * len, items[i].k_offset = items[i].v_offset = i * cache;
                    items[i].sinks_offset = LNG_NO_SINKS, items[i].start = w.ctx - 1 - i, items[i].window = LNG_WINDOW_FULL, items[i].slots = w.ctx;
                }
                auto record = [&] {
                    return table ? lng_hip_attention_decode_batched(f.batch, 0, 1, 2, 3, LNG_NO_SINKS, items, 2, heads, kv, w.dim, 0.125f, LNG_F32)
                                 : lng_hip_attention_grouped(f.batch, lng_slice{0, 0, len}, lng_slice{1, 0, cache}, lng_slice{2, 0, cache}, lng_slice{3, 0, len}, nullptr, &one, LNG_F32);
                };
                lng_null_clear();
                lng_null_fail_malloc_after(nth + table);
                const int rc = record();
                lng_null_fail_malloc_after(0);
                CHECK(rc == (w.whole ? LNG_OK : LNG_ERR_ALLOC) && lng_hip_batch_dispatches(f.batch) == (w.whole ? 1u : 0u));
                if (!w.whole) CHECK(record() == LNG_OK);
                CHECK(lng_hip_batch_commit(f.batch, nullptr, nullptr) == LNG_OK && lng_hip_batch_wait(f.batch, nullptr) == LNG_OK);
                lng_k_attn a{};
                unsigned grid = 0;
                CHECK(launched().size() == (w.whole ? 1u : 2u) && launch_args(0, "lng_decode_f32", &a, &grid));
                if (w.whole) CHECK(launched()[0] == "lng_decode_f32_d64" && a.chunk == 512 && a.n_chunks == 1 && grid == (table ? 2 : 1) * kv);
                else CHECK(a.n_chunks > 1);
            }
        }
    }
    lng_null_clear();
    // Q8_0 products of few positions do without the planes of their positions when there is no memory for them (17 to 31, which
    // prefer lng_q8_mid, ask a second time, which succeeds here)
    for (const uint64_t n : {16, 31}) {
        for (const bool normed : {false, true}) {
            Fixture f(4, 9 << 20);
            const uint64_t rows = 4096, cols = 2048;
            const lng_slice codes{0, 0, rows * cols}, scales{1, 0, rows * cols / 16}, x{2, 0, n * cols * 4}, y{3, 0, n * rows * 4}, norm{2, x.len, cols * 4};
            const lng_q8_matrix m{codes, scales, y, rows};
            lng_null_clear();
            lng_null_fail_malloc_after(1);
            CHECK((normed ? lng_hip_gemm_q8_0_many_normed(f.batch, &m, 1, x, norm, 1e-5f, cols, n, cols) : lng_hip_gemm_q8_0(f.batch, codes, scales, x, y, rows, cols, n, cols, rows)) == LNG_OK);
            lng_null_fail_malloc_after(0);
            CHECK(lng_hip_batch_commit(f.batch, nullptr, nullptr) == LNG_OK && lng_hip_batch_wait(f.batch, nullptr) == LNG_OK);
            CHECK(launched() == (n == 16 ? std::vector<std::string>{"lng_q8_few_f32"} : std::vector<std::string>{"lng_q8_norm_frag", "lng_q8_few"}));
        }
    }
    lng_hip_batch_drop(batch);
    for (lng_buffer *b : bufs) CHECK(lng_hip_buffer_free(b) == LNG_OK);
    lng_hip_close(gpu);
    CHECK(lng_null_live_allocations() == 0);
    lng_null_clear();
}

// ---- the planner fuzz -------------------------------------------------------------------------------------

static uint64_t visible_from_tile(const lng_k_row &r) { // the run a row's chunks cover: from the 32-aligned window start
    const uint64_t last = r.start;
    const uint64_t first = (r.window != LNG_WINDOW_FULL && last + 1 > r.window) ? last + 1 - r.window : 0;
    return last + 1 - (first & ~(uint64_t)31);
}

// The kernels' own search (work_of in lng_kernels.hip) on the host: the row of workgroup w in cum[0..n_rows].
static uint32_t row_of_workgroup(const uint32_t *cum, uint32_t n_rows, uint32_t w) {
    uint32_t lo = 0, n = n_rows;
    while (n > 64u) {
        const uint32_t stride = (n + 63u) / 64u;
        uint32_t cnt = 0;
        for (uint32_t lane = 0; lane < 64; ++lane) cnt += lane * stride < n && cum[lo + lane * stride] <= w;
        const uint32_t step = (cnt - 1u) * stride;
        n = n - step < stride ? n - step : stride;
        lo += step;
    }
    uint32_t cnt = 0;
    for (uint32_t lane = 0; lane < 64; ++lane) cnt += lane < n && cum[lo + lane] <= w;
    return lo + cnt - 1u;
}

struct FuzzStats {
    size_t dispatches = 0, split = 0, fused = 0, tables = 0, generic = 0, wide = 0, prefill = 0;
};

// Checks the launches recorded for ONE dispatch whose rows are `rows` (one per query row).
static void check_rows_dispatch(const std::vector<lng_k_row> &rows, uint32_t heads, uint32_t kv_heads, uint32_t dim, FuzzStats &st) {
    const size_t n_launches = lng_null_launch_count();
    CHECK(n_launches >= 1 && n_launches <= 2);
    const char *name = nullptr;
    unsigned grid[3], block[3];
    const void *args = nullptr;
    size_t args_size = 0;
    CHECK(lng_null_launch(0, &name, grid, block, &args, &args_size) == 0);
    const std::string kernel = name;
    if (kernel.rfind("lng_prefill_", 0) == 0) { // several rows over a long cache: the prompt-pass kernels
        CHECK(args_size == sizeof(lng_k_prefill));
        lng_k_prefill p;
        memcpy(&p, args, sizeof p);
        CHECK(p.splits >= 1 && p.splits <= 64 && p.t == rows.size());
        if (p.splits > 1) {
            const uint64_t slots = p.t * p.heads * p.splits;
            CHECK(lng_null_bytes_from(p.partial_o) >= slots * p.dim * 4);
            CHECK(lng_null_bytes_from(p.partial_ml) >= slots * 2 * 4);
            CHECK(n_launches == 2);
        } else {
            CHECK(n_launches == 1);
        }
        st.prefill += 1;
        return;
    }
    CHECK(args_size == sizeof(lng_k_attn));
    lng_k_attn a;
    memcpy(&a, args, sizeof a);
    CHECK(a.n_rows == rows.size() && a.heads == heads && a.kv_heads == kv_heads && a.dim == dim);
    CHECK(block[0] == 256 && grid[1] == 1 && grid[2] == 1);
    const uint32_t group = heads / kv_heads;
    if (kernel.rfind("lng_attn_generic", 0) == 0) {
        CHECK(grid[0] == rows.size() * heads && n_launches == 1);
        st.generic += 1;
        return;
    }
    if (kernel.find("_w") != std::string::npos) st.wide += 1;
    CHECK(a.chunk >= 128 && a.chunk % 128 == 0 && a.n_chunks >= 1 && a.n_chunks <= LNG_MAX_CHUNKS);
    uint64_t longest = 0, live = 0;
    for (const lng_k_row &r : rows) {
        longest = std::max(longest, visible_from_tile(r));
        live += (visible_from_tile(r) + a.chunk - 1) / a.chunk * kv_heads;
    }
    CHECK((longest + a.chunk - 1) / a.chunk == a.n_chunks); // the partials keep n_chunks slots per (row, kv head)
    const uint64_t pairs = rows.size() * (uint64_t)kv_heads;
    std::vector<uint8_t> taken(pairs * a.n_chunks, 0);
    if (a.work) {
        st.tables += 1;
        CHECK(a.n_chunks > 1 && grid[0] == live);
        CHECK(lng_null_bytes_from(a.work) >= (rows.size() + 1) * 4);
        const uint32_t *cum = a.work; // the null device's device memory is host memory: the table as the kernel reads it
        CHECK(cum[0] == 0 && cum[rows.size()] == grid[0]);
        for (size_t r = 0; r < rows.size(); ++r) {
            CHECK(cum[r + 1] - cum[r] == (visible_from_tile(rows[r]) + a.chunk - 1) / a.chunk * kv_heads);
        }
        for (uint32_t w = 0; w < grid[0]; ++w) {
            const uint32_t row = row_of_workgroup(cum, (uint32_t)rows.size(), w);
            CHECK(row < rows.size() && cum[row] <= w && w < cum[row + 1]);
            const uint32_t chunks = (cum[row + 1] - cum[row]) / kv_heads, local = w - cum[row];
            const uint64_t pair = (uint64_t)row * kv_heads + local / chunks, chunk = local % chunks;
            CHECK(pair < pairs && chunk < a.n_chunks && !taken[pair * a.n_chunks + chunk]);
            taken[pair * a.n_chunks + chunk] = 1;
        }
    } else {
        CHECK(grid[0] == pairs * a.n_chunks);
        for (uint32_t w = 0; w < grid[0]; ++w) taken[w] = 1; // pair w / n_chunks, chunk w % n_chunks
    }
    // every chunk a row has was taken once, and has positions: chunk c of a row's n takes its groups of 128 positions
    // c, c + n, ...: the first of them must start inside the row's run
    for (size_t r = 0; r < rows.size(); ++r) {
        const uint64_t run = visible_from_tile(rows[r]), chunks = (run + a.chunk - 1) / a.chunk;
        for (uint32_t g = 0; g < kv_heads; ++g) {
            for (uint64_t c = 0; c < a.n_chunks; ++c) {
                const bool has = c < chunks;
                if (has) CHECK(taken[(r * kv_heads + g) * a.n_chunks + c] && c * 128 < run);
                if (!has && a.work) CHECK(!taken[(r * kv_heads + g) * a.n_chunks + c]);
            }
        }
    }
    if (a.n_chunks > 1) {
        st.split += 1;
        const uint64_t slots = pairs * a.n_chunks * group;
        CHECK(lng_null_bytes_from(a.partial_o) >= slots * dim * 4);
        CHECK(lng_null_bytes_from(a.partial_ml) >= slots * 2 * 4);
        if (a.fused) {
            st.fused += 1;
            CHECK(lng_null_bytes_from(a.tickets) >= pairs * 4 && n_launches == 1);
            for (uint64_t i = 0; i < pairs; ++i) CHECK(a.tickets[i] == 0); // zero whenever no dispatch is running
        } else {
            CHECK(n_launches == 2);
            const char *merge = nullptr;
            unsigned mgrid[3];
            CHECK(lng_null_launch(1, &merge, mgrid, nullptr, nullptr, nullptr) == 0);
            const std::string m = merge;
            CHECK(m == "lng_decode_merge" || m == "lng_decode_merge_few");
            CHECK(mgrid[0] == (m == "lng_decode_merge" ? pairs * group : pairs * ((group + 3) / 4)));
            if (m == "lng_decode_merge_few") CHECK(a.n_chunks <= 32);
        }
    } else {
        CHECK(n_launches == 1 && !a.fused);
    }
}

static void planner_fuzz(size_t dispatches) {
    std::mt19937_64 rng(20251125);
    auto below = [&](uint64_t n) { return (uint64_t)(rng() % n); };
    lng_gpu *gpu = nullptr;
    CHECK(lng_hip_open(0, &gpu) == LNG_OK);
    // one big cache for every row (inputs may share; outputs may not)
    const uint64_t max_rows = 70000;
    const size_t kv_bytes = max_rows * 2 * 64 * 4, qo_bytes = (size_t)300 * 160 * 512 * 4; // the most rows x heads x width x 4 drawn below
    std::vector<lng_buffer *> bufs(5);
    const size_t sizes[5] = {qo_bytes, kv_bytes, kv_bytes, qo_bytes, 4096};
    for (int i = 0; i < 5; ++i) CHECK(lng_hip_buffer(gpu, sizes[i], &bufs[i]) == LNG_OK);
    FuzzStats st;
    const uint32_t dims[] = {64, 64, 64, 64, 128, 256, 512, 96, 32};
    for (size_t it = 0; it < dispatches; ++it) {
        lng_batch *batch = nullptr;
        CHECK(lng_hip_batch(gpu, bufs.data(), bufs.size(), &batch) == LNG_OK);
        const uint32_t dim = dims[below(9)];
        const uint32_t kv_heads = 1u << below(dim >= 256 ? 2 : 4); // 1..8
        const uint32_t group = (uint32_t)(1 + below(below(8) == 0 ? 20 : 8));
        const uint32_t heads = kv_heads * group;
        const int dtype = below(4) == 0 ? LNG_F32 : LNG_BF16;
        const uint64_t es = dtype == LNG_F32 ? 4 : 2, row_bytes = (uint64_t)kv_heads * dim * es, qrow = (uint64_t)heads * dim * es;
        const uint64_t most = std::min<uint64_t>(max_rows, kv_bytes / row_bytes);
        // lengths: mostly short, sometimes long, sometimes all alike
        auto length = [&]() -> uint64_t {
            switch (below(6)) {
            case 0: return 1 + below(160);
            case 1: return 1 + below(most);
            case 2: return 128 * (1 + below(64));
            default: return 1 + below(9000);
            }
        };
        std::vector<lng_k_row> rows;
        int rc;
        if (below(3) == 0) { // the row-by-row operator: t consecutive rows of one cache
            const uint64_t t = 1 + below(below(4) == 0 ? 40 : 4);
            const uint64_t end = std::min<uint64_t>(most, std::max<uint64_t>(length(), t));
            const uint64_t start = end - t;
            uint64_t window = below(3) == 0 ? 1 + below(3000) : LNG_WINDOW_FULL;
            uint64_t slots = end;
            if (window != LNG_WINDOW_FULL && below(2) == 0) slots = std::min<uint64_t>(end, window + t + below(64)); // a ring
            const lng_grouped_shape s = shape(t, start, heads, kv_heads, dim, window, slots, 0.125f);
            const uint64_t kv_rows = std::min(slots, end);
            const uint64_t off = below(4) == 0 ? es * (1 + below(3)) : 0; // sometimes off a 16-byte boundary
            const lng_slice q{0, off, t * qrow}, k{1, 0, kv_rows * row_bytes}, v{2, 0, kv_rows * row_bytes}, o{3, 0, t * qrow}, sk{4, 0, heads * 4ull};
            rc = lng_hip_attention_grouped(batch, q, k, v, o, below(2) ? &sk : nullptr, &s, dtype);
            if (dim % 32 != 0) {
                CHECK(rc == LNG_ERR_DISPATCH);
            } else {
                CHECK(rc == LNG_OK);
            }
            for (uint64_t i = 0; i < t; ++i) rows.push_back(lng_k_row{0, 0, 0, 0, 0, start + i, window, slots});
        } else { // a table of sequences
            const size_t n = 1 + below(below(5) == 0 ? 300 : 40);
            std::vector<lng_decode_item> items(n);
            const bool alike = below(5) == 0;
            const uint64_t same = length();
            for (size_t i = 0; i < n; ++i) {
                const uint64_t len = std::min<uint64_t>(most, alike ? same : length());
                const uint64_t window = below(4) == 0 ? 1 + below(2000) : LNG_WINDOW_FULL;
                uint64_t slots = len;
                if (window != LNG_WINDOW_FULL && below(2) == 0) slots = std::min<uint64_t>(len, window + 1 + below(32));
                items[i] = lng_decode_item{i * qrow, i * qrow, 0, 0, below(2) ? 0 : LNG_NO_SINKS, len - 1, window, slots};
                rows.push_back(items[i]);
            }
            rc = lng_hip_attention_decode_batched(batch, 0, 1, 2, 3, 4, items.data(), n, heads, kv_heads, dim, 0.125f, dtype);
            if (dim % 32 != 0) {
                CHECK(rc == LNG_ERR_DISPATCH);
            } else {
                CHECK(rc == LNG_OK);
            }
        }
        if (rc == LNG_OK) {
            CHECK(lng_hip_batch_commit(batch, nullptr, nullptr) == LNG_OK);
            CHECK(lng_hip_batch_wait(batch, nullptr) == LNG_OK);
            check_rows_dispatch(rows, heads, kv_heads, dim, st);
            st.dispatches += 1;
        }
        lng_hip_batch_drop(batch);
        lng_null_clear();
        if (g_failures) {
            fprintf(stderr, "fuzz dispatch %zu: %zu rows, %u heads over %u of width %u, dtype %d\n", it, rows.size(), heads, kv_heads, dim, dtype);
            break;
        }
    }
    for (lng_buffer *b : bufs) CHECK(lng_hip_buffer_free(b) == LNG_OK);
    lng_hip_close(gpu);
    CHECK(lng_null_live_allocations() == 0);
    printf("planner fuzz: %zu dispatches checked (%zu split, %zu merged in the kernel, %zu with a table of live workgroups, %zu on the "
           "generic kernel, %zu at widths 128-512, %zu on a prompt-pass kernel)\n",
           st.dispatches, st.split, st.fused, st.tables, st.generic, st.wide, st.prefill);
    CHECK(st.split > st.dispatches / 20 && st.fused > 0 && st.tables > 0 && st.generic > 0 && st.wide > 0 && st.prefill > 0);
}

int main(int argc, char **argv) {
    const size_t dispatches = argc > 1 ? (size_t)strtoull(argv[1], nullptr, 10) : 100000;
    refusals();
    products_and_their_kernels();
    fused_sequences();
    switches_and_checksum();
    lifetimes();
    allocation_failures();
    planner_fuzz(dispatches);
    if (g_failures) {
        fprintf(stderr, "%d checks failed\n", g_failures);
        return 1;
    }
    printf("null device: all checks held\n");
    return 0;
}
