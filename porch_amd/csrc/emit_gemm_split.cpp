// fp32 products on the bf16 matrix cores, at fp32 accuracy.
//
// The fp32 MFMA of gfx950 runs at a sixteenth of the bf16 one's rate (157
// against 2517 TFLOP/s).  Every fp32 value is the sum of three bf16 values,
// x = h + m + l with h = bf16(x), m = bf16(x - h), l = x - h - m: both
// differences are exact, and l has at most eight significant bits.  Of the
// nine products of two such sums the kernel takes the six above 2^-26 of
// the whole (hh, mh, hm, mm, lh, hl), each exact in fp32, and sums them in
// the MFMA's fp32 accumulators.  What is left out is below half an ulp of
// each product, and one MFMA adds 16 products to the accumulator with one
// rounding where the fp32 MFMA adds two.  Relative error (2-norm) against
// 64 bits, one tile, this form / the fp32 MFMA: N(0,1) operands, K = 16
// 6.0e-8 / 8.2e-8 (fewer values of K stay on the fp32 MFMA), K = 64 1.1e-7 /
// 1.4e-7, K = 1024 4.9e-7 / 5.4e-7, K = 4096 1.04e-6 / 1.23e-6, K = 16384
// 2.25e-6 / 2.32e-6; U(0,1), K = 4096 5.3e-7 / 8.5e-7.
//
// Values the split cannot hold exactly send a tile to the fp32 MFMA, in the
// same kernel (`redo` below):
//   - infinities, NaN and values that round to an infinite bf16: every one
//     of them makes its whole row or column of the tile NaN (inf - inf in
//     the split), and so does a sum that overflows; a tile with a result
//     that is not finite is computed again;
//   - nonzero values below 2^-109, whose last bits bf16 (down to 2^-133)
//     drops: what is lost is at most 2^-133 times the other operand per
//     product.  With the operands below 2^30 and K below 2^20 that is below
//     2^-83, so results of 2^-56 and more keep their accuracy; a tile that
//     read such a value and has a smaller result or a larger operand is
//     computed again.
//
// What bounds it: at 4096^3 the rate is that of this card's large bf16
// products (1.39 PFLOP/s of bf16 products against 1.34-1.42 measured for
// the vendor library's bf16 product of the same size), which its power
// limits.  Below that size a tile's step is a chain (loads, split, LDS,
// MFMA) that eight waves on a compute unit overlap.

#include "emit_gemm.hpp"

#include <algorithm>
#include <stdexcept>

namespace porch::cg {

    namespace {

        // Eight waves a workgroup, one workgroup a compute unit.  256 x 256
        // tiles (waves of 128 x 64, K in steps of 16): the fewest LDS reads
        // and splits per MFMA.  128 x 128 tiles (waves of 32 x 64, K in
        // steps of 32, so that a step's fixed costs cover as many MFMAs):
        // four times the workgroups.
        struct tiling {
            int bm, bn;        // output tile
            int ks;            // 16-wide slices of K per step
            int wms, wns;      // waves along m, n
            [[nodiscard]] int bk() const { return 16 * ks; }
        };
        constexpr tiling LARGE{256, 256, 1, 2, 4};
        constexpr tiling SMALL{128, 128, 2, 4, 2};
        constexpr int THREADS = 512;

        // A round of 256 x 256 tiles over the compute units takes 3.2 times
        // as long as one of 128 x 128 (K of 1024: 156 us for one against
        // 191 us for four rounds), so the large tile pays where it saves
        // more rounds than that.
        const tiling& choose(const gemm_request& r) {
            const int64_t cus = std::max(r.compute_units, 8);
            auto rounds = [&](const tiling& t) {
                const int64_t tiles = ((r.m + t.bm - 1) / t.bm) * ((r.n + t.bn - 1) / t.bn) * r.batch;
                return (tiles + cus - 1) / cus;
            };
            return r.k_chunks == 1 && 16 * rounds(LARGE) < 5 * rounds(SMALL) ? LARGE : SMALL;
        }

        // How an operand's tile is read.  `rows`: along its m (A) or n (B).
        enum class reading {
            along_k,    // contiguous along K: four values of a row, 128 bits
            along_rows, // contiguous along the rows: two rows, four loads of 64 bits
            strided     // neither: four values of a row, 32 bits each
        };

        struct operand_tile {
            std::string x;             // "A" or "B"
            std::string origin;        // "m0" or "n0"
            int rows;                  // of the tile
            int64_t extent;            // of the matrix
            int64_t stride_row, stride_k;
            reading how;
            int units;                 // per thread
        };

        operand_tile tile_of(const gemm_request& r, const tiling& t, bool is_a) {
            const gemm_operand& op = is_a ? r.a : r.b;
            operand_tile o;
            o.x = is_a ? "A" : "B";
            o.origin = is_a ? "m0" : "n0";
            o.rows = is_a ? t.bm : t.bn;
            o.extent = is_a ? r.m : r.n;
            o.stride_row = is_a ? op.stride_row : op.stride_col;
            o.stride_k = is_a ? op.stride_col : op.stride_row;
            // 64- and 128-bit loads need 4-byte alignment only (gfx950 reads
            // unaligned vectors), so offsets and odd strides don't matter
            if (o.stride_k == 1) o.how = reading::along_k;
            else if (o.stride_row == 1 && o.extent >= 2) o.how = reading::along_rows;
            else o.how = reading::strided;
            const int values = o.how == reading::along_rows ? 8 : 4;
            o.units = o.rows * t.bk() / values / THREADS;
            return o;
        }

        // Byte offsets: 32 bits where every tensor has fewer than 2^30
        // elements, so that a load is one instruction over a scalar base.
        const char* offset_type(const gemm_request& r) { return r.width.wide ? "long long" : "unsigned"; }

        // Per-thread constants of an operand's loads: byte offset o{X}{i} of
        // unit i at k = 0 of a step, its first k kq{X}{i}, and the LDS row it
        // is written to.
        std::string setup_code(const gemm_request& r, const tiling& t, const operand_tile& o) {
            std::string s;
            const std::string R = std::to_string(o.rows), OT = offset_type(r);
            const std::string shift = std::to_string(t.ks == 1 ? 8 : 4);
            for (int i = 0; i < o.units; ++i) {
                const std::string id = o.x + std::to_string(i);
                s += "    const int c" + id + " = tid + " + std::to_string(i * THREADS) + ";\n";
                if (o.how == reading::along_rows) {
                    // lanes: two halves of an octet of k, then pairs of rows
                    s += "    const int oct" + id + " = (c" + id + " >> 1) / " + std::to_string(o.rows / 2) + ";\n";
                    s += "    const int kq" + id + " = oct" + id + " * 8 + (c" + id + " & 1) * 4;\n";
                    s += "    const int i" + id + " = ((c" + id + " >> 1) % " + std::to_string(o.rows / 2) + ") * 2;\n";
                    s += "    const int p" + id + " = (i" + id + " & ~63) | ((i" + id + " >> 1) & 31);\n";
                    s += "    const idx_t g" + id + " = " + o.origin + " + i" + id + " < " + std::to_string(o.extent - 2) +
                         " ? " + o.origin + " + i" + id + " : (idx_t)" + std::to_string(o.extent - 2) + ";\n";
                    // the last row of an odd extent is the second of its pair
                    if (o.extent % 2 != 0)
                        s += "    const bool last" + id + " = " + o.origin + " + i" + id + " == " +
                             std::to_string(o.extent - 1) + ";\n";
                }
                else {
                    const std::string per_row = std::to_string(t.bk() / 4);
                    s += "    const int kq" + id + " = (c" + id + " % " + per_row + ") * 4;\n";
                    s += "    const int oct" + id + " = kq" + id + " >> 3;\n";
                    s += "    const int p" + id + " = c" + id + " / " + per_row + ";\n";
                    s += "    const idx_t i" + id + " = " + o.origin + " + porch_row(p" + id + ");\n";
                    s += "    const idx_t g" + id + " = i" + id + " < " + std::to_string(o.extent) + " ? i" + id +
                         " : (idx_t)" + std::to_string(o.extent - 1) + ";\n";
                }
                s += "    const " + OT + " o" + id + " = ((" + OT + ")g" + id + " * " + std::to_string(o.stride_row) +
                     " + (" + OT + ")kq" + id + " * " + std::to_string(o.stride_k) + ") * 4;\n";
                s += "    const int w" + id + " = (((oct" + id + " >> 1) * 2 + (oct" + id + " & 1)) * " + R + " + (p" + id +
                     " ^ (oct" + id + " * " + shift + "))) * 12 + ((kq" + id + " >> 2) & 1) * 2;\n";
            }
            s += "    float r" + o.x + "[" + std::to_string(o.units * (o.how == reading::along_rows ? 8 : 4)) + "];\n";
            return s;
        }

        // Loads the operand's values of the step at element `k0` of K into
        // registers; `tail`: only the first `tail` values of K exist (the
        // rest read as zero).
        std::string load_code(const operand_tile& o, const std::string& k0, int64_t tail, const std::string& ind) {
            std::string s;
            const std::string SK = std::to_string(o.stride_k);
            s += ind + "{\n" + ind + "    const char* __restrict__ base = (const char*)(" + o.x + " + (idx_t)(" + k0 + ") * " +
                 SK + ");\n";
            for (int i = 0; i < o.units; ++i) {
                const std::string id = o.x + std::to_string(i);
                const int at = i * (o.how == reading::along_rows ? 8 : 4);
                auto reg = [&](int j) { return "r" + o.x + "[" + std::to_string(at + j) + "]"; };
                if (o.how == reading::along_k && tail == 0) {
                    s += ind + "    const porch_f4u v" + id + " = *(const porch_f4u*)(base + o" + id + ");\n" + ind + "    ";
                    const char* e[] = {"x", "y", "z", "w"};
                    for (int j = 0; j < 4; ++j) s += reg(j) + " = v" + id + "." + e[j] + "; ";
                    s += "\n";
                    continue;
                }
                for (int j = 0; j < 4; ++j) {
                    const std::string J = std::to_string(j);
                    const std::string p = "(base + o" + id + " + " + std::to_string(j * o.stride_k * 4) + "LL)";
                    const std::string guard = tail == 0 ? "" : "kq" + id + " + " + J + " < " + std::to_string(tail);
                    if (o.how == reading::along_rows) {
                        s += ind + "    porch_f2u v" + id + J + " = {0.0f, 0.0f};\n";
                        s += ind + "    " + (tail ? "if (" + guard + ") " : "") + "v" + id + J + " = *(const porch_f2u*)" + p + ";\n";
                        s += ind + "    " + reg(j) + " = " +
                             (o.extent % 2 != 0 ? "last" + id + " ? v" + id + J + ".y : " : std::string()) + "v" + id + J +
                             ".x; " + reg(4 + j) + " = v" + id + J + ".y;\n";
                    }
                    else {
                        s += ind + "    " + reg(j) + " = " + (tail ? guard + " ? " : std::string()) + "*(const float*)" + p +
                             (tail ? " : 0.0f" : "") + ";\n";
                    }
                }
            }
            return s + ind + "}\n";
        }

        std::string store_code(const operand_tile& o, const std::string& buffer, const std::string& ind) {
            std::string s;
            for (int i = 0; i < o.units; ++i) {
                const std::string id = o.x + std::to_string(i);
                const int at = i * (o.how == reading::along_rows ? 8 : 4);
                for (int e = 0; e < (o.how == reading::along_rows ? 2 : 1); ++e) {
                    s += ind + "porch_split4(";
                    for (int j = 0; j < 4; ++j) s += "r" + o.x + "[" + std::to_string(at + 4 * e + j) + "], ";
                    s += "&" + o.x + "s[" + buffer + "][0][0][0] + w" + id + (e ? " + 384" : "") + ", lowest, largest);\n";
                }
            }
            return s;
        }

    } // namespace

    const char* bf16_split_helpers() {
        return R"(typedef float porch_v16f __attribute__((ext_vector_type(16)));
typedef float porch_v2f __attribute__((ext_vector_type(2)));
typedef float porch_f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float porch_f2u __attribute__((ext_vector_type(2), aligned(4)));
typedef __bf16 porch_b2 __attribute__((ext_vector_type(2)));
typedef __bf16 porch_b8 __attribute__((ext_vector_type(8)));
typedef unsigned porch_u2 __attribute__((ext_vector_type(2)));
typedef unsigned short porch_s2 __attribute__((ext_vector_type(2)));
// Row of the tile held at LDS row p: pairs of adjacent rows lie 32 apart, so
// that a lane's two MFMA blocks cover two adjacent rows (columns of C).
__device__ __forceinline__ int porch_row(int p) { return (p & ~63) | ((p & 31) << 1) | ((p >> 5) & 1); }
__device__ __forceinline__ unsigned porch_bf16_pair(float x, float y) {
    const porch_v2f v = {x, y};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, porch_b2));
}
// Two values as bf16 pairs h + m + l, exactly.
__device__ __forceinline__ void porch_split2(float x, float y, unsigned& h, unsigned& m, unsigned& l) {
    h = porch_bf16_pair(x, y);
    const float rx = x - __builtin_bit_cast(float, h << 16), ry = y - __builtin_bit_cast(float, h & 0xffff0000u);
    m = porch_bf16_pair(rx, ry);
    l = porch_bf16_pair(rx - __builtin_bit_cast(float, m << 16), ry - __builtin_bit_cast(float, m & 0xffff0000u));
}
// The same, noting the least of 2 |bits| - 1 (zeros as the greatest) and the
// largest |h|.
__device__ __forceinline__ void porch_split2(float x, float y, unsigned& h, unsigned& m, unsigned& l, unsigned& lowest,
                                             porch_s2& largest) {
    const unsigned ux = (__builtin_bit_cast(unsigned, x) << 1) - 1u, uy = (__builtin_bit_cast(unsigned, y) << 1) - 1u;
    const unsigned u = ux < uy ? ux : uy;
    lowest = u < lowest ? u : lowest;
    porch_split2(x, y, h, m, l);
    largest = __builtin_elementwise_max(largest, __builtin_bit_cast(porch_s2, h & 0x7fff7fffu));
}
__device__ __forceinline__ void porch_split4(float a, float b, float c, float d, float* to, unsigned& lowest,
                                             porch_s2& largest) {
    porch_u2 h, m, l;
    unsigned hx, hy, mx, my, lx, ly;
    porch_split2(a, b, hx, mx, lx, lowest, largest);
    porch_split2(c, d, hy, my, ly, lowest, largest);
    h.x = hx; h.y = hy; m.x = mx; m.y = my; l.x = lx; l.y = ly;
    *(porch_u2*)to = h;
    *(porch_u2*)(to + 4) = m;
    *(porch_u2*)(to + 8) = l;
}
)";
    }

    kernel_code emit_gemm_split(const gemm_request& r) {
        const tiling& t = choose(r);
        const int BK = t.bk();
        const operand_tile A = tile_of(r, t, true);
        const operand_tile B = tile_of(r, t, false);
        const int64_t tiles_m = (r.m + t.bm - 1) / t.bm;
        const int64_t tiles_n = (r.n + t.bn - 1) / t.bn;
        const int64_t tiles = tiles_m * tiles_n;
        const int64_t total = tiles * r.batch;
        const int64_t chunks = r.k_chunks;
        // Steps in the order they run: a partial last one (masked loads)
        // first, so that the loop's loads need no tests.
        const int64_t full = r.k / BK;
        const int64_t tail = r.k % BK;
        const int64_t steps = full + (tail != 0 ? 1 : 0);
        if (chunks > 1 && steps < 2 * chunks) throw std::logic_error("emit_gemm_split: chunks of two steps or more");
        const int wave_m = t.bm / t.wms, wave_n = t.bn / t.wns;
        const int ib = wave_m / 32, jb = wave_n / 32;
        const std::string IB = std::to_string(ib), JB = std::to_string(jb);
        const std::string M = std::to_string(r.m), N = std::to_string(r.n);
        const std::string WM = std::to_string(wave_m), WN = std::to_string(wave_n);
        const std::string BM = std::to_string(t.bm), BN = std::to_string(t.bn);

        kernel_code kc;
        kc.kind = "gemm.mfma";
        kc.name = "porch_gemm";
        kc.n_slots = r.n_slots;
        kc.block = THREADS;
        kc.grid_x = static_cast<unsigned>(total * chunks);
        std::string& s = kc.source;
        s = kernel_prologue(r.n_slots, r.width.type());
        s += bf16_split_helpers();
        s += "extern \"C\" __global__ void __launch_bounds__(512, 2) porch_gemm(" + kernel_params(r.n_slots) + ") {\n";
        // [buffer][slice of 16][octet of k, row][h, m, l: 8 bf16 each].  With
        // the 48-byte pitch 16 consecutive rows meet every bank once per
        // 128-bit read; the rows of octet o are stored at row ^ 8 o (4 o with
        // four octets a step), so that the octets of one row that adjacent
        // lanes write do too.
        s += "    __shared__ __attribute__((aligned(16))) float As[2][" + std::to_string(t.ks) + "][" +
             std::to_string(2 * t.bm) + "][12];\n";
        s += "    __shared__ __attribute__((aligned(16))) float Bs[2][" + std::to_string(t.ks) + "][" +
             std::to_string(2 * t.bn) + "][12];\n";
        s += "    __shared__ unsigned seen[8];\n";
        s += "    const int tid = threadIdx.x;\n    const int lane = tid & 63;\n    const int wave = tid >> 6;\n";
        s += "    const int wm = wave / " + std::to_string(t.wns) + ";\n    const int wn = wave % " +
             std::to_string(t.wns) + ";\n";
        // Workgroups are dispatched round-robin over the 8 XCDs; each XCD
        // takes a contiguous run of (entry, tile) pairs, so that its L2 holds
        // their panels.  (The chunks of a split K keep the plain order.)
        if (chunks > 1) {
            s += "    const int chunk = blockIdx.x % " + std::to_string(chunks) + ";\n";
            s += "    const idx_t lin = blockIdx.x / " + std::to_string(chunks) + ";\n";
            s += "    const int g0 = (int)((long long)chunk * " + std::to_string(steps) + " / " + std::to_string(chunks) + ");\n";
            s += "    const int g1 = (int)((long long)(chunk + 1) * " + std::to_string(steps) + " / " + std::to_string(chunks) + ");\n";
        }
        else {
            const int64_t each = total / 8, more = total % 8;
            s += "    const int xcd = blockIdx.x % 8;\n";
            s += "    const idx_t lin = (idx_t)xcd * " + std::to_string(each) +
                 (more ? " + (xcd < " + std::to_string(more) + " ? xcd : " + std::to_string(more) + ")" : std::string()) +
                 " + blockIdx.x / 8;\n";
            s += "    const int g0 = 0;\n    const int g1 = " + std::to_string(steps) + ";\n";
        }
        if (r.batched) s += "    const idx_t qb = lin / " + std::to_string(tiles) + ";\n";
        s += "    const int tile = (int)(lin" + (r.batched ? " % " + std::to_string(tiles) : std::string()) + ");\n";
        s += "    const idx_t m0 = (idx_t)(tile / " + std::to_string(tiles_n) + ") * " + BM + ";\n";
        s += "    const idx_t n0 = (idx_t)(tile % " + std::to_string(tiles_n) + ") * " + BN + ";\n";
        auto base = [&](const char* x, const gemm_operand& op) {
            s += std::string("    const float* __restrict__ ") + x + " = a" + std::to_string(op.slot) + " + " +
                 std::to_string(op.offset);
            if (r.batched && op.stride_batch != 0) s += " + qb * " + std::to_string(op.stride_batch);
            s += ";\n";
        };
        base("A", r.a);
        base("B", r.b);
        s += setup_code(r, t, A) + setup_code(r, t, B);
        s += "    unsigned lowest = 0xffffffffu;\n    porch_s2 largest = {0, 0};\n";
        s += "    porch_v16f acc[" + IB + "][" + JB + "];\n";
        const std::string zero_acc =
            "    #pragma unroll\n    for (int i = 0; i < " + IB + "; ++i)\n        #pragma unroll\n        for (int j = 0; j < " +
            JB + "; ++j)\n            #pragma unroll\n            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;\n";
        s += zero_acc;

        auto load_both = [&](const std::string& k0, int64_t masked, const std::string& ind) {
            return load_code(A, k0, masked, ind) + load_code(B, k0, masked, ind);
        };
        auto store_both = [&](const std::string& buffer, const std::string& ind) {
            return store_code(A, buffer, ind) + store_code(B, buffer, ind);
        };
        auto whole = [&](const std::string& g) {
            return "(" + g + (tail != 0 ? " - 1" : "") + ") * " + std::to_string(BK);
        };
        // prologue: the first step in LDS, the second in registers
        const std::string partial = std::to_string(full * BK);
        if (tail != 0 && chunks > 1)
            // the first chunk alone holds the partial step
            s += "    if (g0 == 0) {\n" + load_both(partial, tail, "        ") + "    }\n    else {\n" +
                 load_both(whole("g0"), 0, "        ") + "    }\n";
        else if (tail != 0)
            s += load_both(partial, tail, "    ");
        else
            s += load_both(whole("g0"), 0, "    ");
        s += store_both("0", "    ");
        if (steps > 1) s += load_both(whole("(g0 + 1)"), 0, "    ");
        s += "    __syncthreads();\n";

        const std::string shift = t.ks == 1 ? "8" : "4";
        auto compute = [&](const std::string& ind) {
            std::string c;
            for (int k = 0; k < t.ks; ++k) {
                const std::string K = std::to_string(k);
                c += ind + "{\n";
                c += ind + "    const int sw = ((lane >> 5) + " + std::to_string(2 * k) + ") * " + shift + ";\n";
                c += ind + "    const int row = (lane & 31) ^ sw;\n";
                c += ind + "    porch_b8 a[3][" + IB + "], b[3][" + JB + "];\n";
                c += ind + "    #pragma unroll\n" + ind + "    for (int p = 0; p < 3; ++p) {\n";
                c += ind + "        #pragma unroll\n" + ind + "        for (int i = 0; i < " + IB + "; ++i) a[p][i] = *(const porch_b8*)&As[cb][" +
                     K + "][(lane >> 5) * " + BM + " + wm * " + WM + " + i * 32 + row][p * 4];\n";
                c += ind + "        #pragma unroll\n" + ind + "        for (int j = 0; j < " + JB + "; ++j) b[p][j] = *(const porch_b8*)&Bs[cb][" +
                     K + "][(lane >> 5) * " + BN + " + wn * " + WN + " + j * 32 + row][p * 4];\n";
                c += ind + "    }\n";
                constexpr int pairs[6][2] = {{0, 0}, {1, 0}, {0, 1}, {1, 1}, {2, 0}, {0, 2}};
                for (const auto& pr : pairs)
                    c += ind + "    #pragma unroll\n" + ind + "    for (int i = 0; i < " + IB + "; ++i)\n" + ind +
                         "        #pragma unroll\n" + ind + "        for (int j = 0; j < " + JB +
                         "; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[" + std::to_string(pr[0]) +
                         "][i], b[" + std::to_string(pr[1]) + "][j], acc[i][j], 0, 0, 0);\n";
                c += ind + "}\n";
            }
            return c;
        };
        if (steps > 1) {
            // One basic block a step: its MFMAs, the split and LDS stores of
            // the next step and the loads of the one after, interleaved by
            // the scheduler (the last steps reload the last one: in bounds,
            // and never used).  With a branch around the stores and loads the
            // 768 x 1024 x 3072 product took 58.8 us against 36.8.
            s += "    for (int g = g0; g < g1; ++g) {\n";
            s += "        const int cb = (g - g0) & 1;\n        const int nb = cb ^ 1;\n";
            s += compute("        ");
            s += store_both("nb", "        ");
            s += "        const int ahead = g + 2 < g1 ? g + 2 : g1 - 1;\n";
            s += load_both(whole("ahead"), 0, "        ");
            s += "        __builtin_amdgcn_iglp_opt(0);\n        __syncthreads();\n    }\n";
        }
        else {
            s += "    {\n        const int cb = 0;\n" + compute("        ") + "    }\n";
        }

        // What the split could not hold (see the top of this file).
        s += "    bool wrong = false, small = false;\n";
        s += "    #pragma unroll\n    for (int i = 0; i < " + IB + "; ++i)\n        #pragma unroll\n        for (int j = 0; j < " +
             JB + "; ++j)\n            #pragma unroll\n            for (int v = 0; v < 16; ++v) {\n";
        s += "                const float x = __builtin_fabsf(acc[i][j][v]);\n";
        s += "                wrong |= !(x <= PORCH_FLT_MAX);\n                small |= !(x >= 0x1p-56f);\n            }\n";
        s += "    const unsigned found = (__ballot(wrong) != 0 ? 1u : 0u) | (__ballot(small || largest.x >= 0x4e80 || "
             "largest.y >= 0x4e80) != 0 ? 2u : 0u) |\n"
             "                           (__ballot(lowest < 0x12000000u) != 0 ? 4u : 0u);\n";
        s += "    if (lane == 0) seen[wave] = found;\n    __syncthreads();\n";
        s += "    unsigned all = 0;\n    #pragma unroll\n    for (int w = 0; w < 8; ++w) all |= seen[w];\n";
        s += "    const bool redo = (all & 1u) != 0 || (all & 6u) == 6u;\n";
        s += "    if (redo) {\n" + zero_acc;
        auto redo_loop = [&](const std::string& lo, const std::string& hi, bool guarded) {
            const std::string K = std::to_string(r.k);
            std::string c = "        for (idx_t k = " + lo + "; k < " + hi + "; k += 2) {\n";
            c += "            const idx_t kk = k + (lane >> 5);\n";
            auto value = [&](const operand_tile& o, const std::string& w, const std::string& extent) {
                std::string l = "            float " + w + "[" + (o.x == "A" ? IB : JB) + "];\n";
                l += "            #pragma unroll\n            for (int i = 0; i < " + (o.x == "A" ? IB : JB) + "; ++i) {\n";
                l += "                const idx_t q = " + o.origin + " + porch_row(" +
                     (o.x == "A" ? "wm * " + WM : "wn * " + WN) + " + i * 32 + (lane & 31));\n";
                l += "                const idx_t at = (q < " + extent + " ? q : (idx_t)" + extent + " - 1) * " +
                     std::to_string(o.stride_row) + " + kk * " + std::to_string(o.stride_k) + ";\n";
                l += "                " + w + "[i] = " + (guarded ? "kk < " + K + " ? " : std::string()) + o.x + "[at]" +
                     (guarded ? " : 0.0f" : "") + ";\n            }\n";
                return l;
            };
            c += value(A, "av", M) + value(B, "bv", N);
            c += "            #pragma unroll\n            for (int i = 0; i < " + IB + "; ++i)\n                #pragma unroll\n"
                 "                for (int j = 0; j < " + JB +
                 "; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i], bv[j], acc[i][j], 0, 0, 0);\n        }\n";
            return c;
        };
        if (full > 0) {
            const std::string lo = tail != 0 ? "(g0 > 0 ? g0 - 1 : 0)" : "g0";
            const std::string hi = tail != 0 ? "(g1 - 1)" : "g1";
            s += redo_loop("(idx_t)" + lo + " * " + std::to_string(BK), "(idx_t)" + hi + " * " + std::to_string(BK), false);
        }
        if (tail != 0) {
            s += "        if (g0 == 0) {\n" + redo_loop(std::to_string(full * BK), std::to_string(r.k), true) + "        }\n";
        }
        s += "    }\n";

        // Epilogue: a lane's blocks 2 j and 2 j + 1 are two adjacent columns.
        const bool m_exact = r.m % t.bm == 0, n_exact = r.n % t.bn == 0;
        auto column = [&](const std::string& to, const std::string& acc, const std::string& q1) {
            if (chunks > 1) return "            const float " + to + " = " + acc + ";\n";
            std::string e = "            float " + to + ";\n            {\n                const float acc_v = " + acc +
                            ";\n                const idx_t q1 = " + q1 + ";\n                (void)q1;\n";
            std::string body;
            emitter em(*r.expr, body, 1);
            em.indent = "                ";
            em.declare_roots({r.epilogue});
            epilogue_emitter(em, r, r.batched ? std::vector<std::string>{"qb", "q0", "q1"} : std::vector<std::string>{"q0", "q1"},
                             "acc_v");
            const std::string v = em.emit(r.epilogue)[0];
            return e + body + "                " + to + " = " + v + ";\n            }\n";
        };
        s += "    #pragma unroll\n    for (int i = 0; i < " + IB + "; ++i)\n    #pragma unroll\n    for (int v = 0; v < 16; ++v) {\n";
        s += "        const idx_t q0 = m0 + porch_row(wm * " + WM + " + i * 32 + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3));\n";
        s += "        #pragma unroll\n        for (int j = 0; j < " + JB + "; j += 2) {\n";
        s += "            const idx_t qn = n0 + wn * " + WN + " + j * 32 + 2 * (lane & 31);\n";
        std::string at = (r.batched ? "(qb * " + M + " + q0) * " : "q0 * ") + N + " + qn";
        if (chunks > 1) at = "chunk * (idx_t)" + std::to_string(r.batch * r.m * r.n) + " + " + at;
        s += "            float* const to = out + " + at + ";\n";
        std::string both;
        if (!m_exact) both = "q0 < " + M;
        if (!n_exact) both += (both.empty() ? "" : " && ") + std::string("qn + 1 < ") + N;
        if (!both.empty()) s += "            if (" + both + ") {\n";
        s += column("x", "acc[i][j][v]", "qn") + column("y", "acc[i][j + 1][v]", "qn + 1");
        s += "            porch_f2u xy = {x, y};\n            *(porch_f2u*)to = xy;\n";
        if (!both.empty()) s += "            }\n";
        if (!n_exact && r.n % 2 != 0) {
            s += "            else if (" + (m_exact ? std::string() : "q0 < " + M + " && ") + "qn < " + N + ") {\n";
            s += column("x", "acc[i][j][v]", "qn") + "            *to = x;\n            }\n";
        }
        s += "        }\n    }\n}\n";
        return kc;
    }

} // namespace porch::cg
