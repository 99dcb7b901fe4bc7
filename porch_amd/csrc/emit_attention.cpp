// softmax(f(Q K), last axis) V in one kernel: the scores never reach memory.
//
// Unfused, the product of 16 heads over 4096 positions writes 1 GiB of
// scores, the softmax reads and writes them and the second product reads
// them again: 1186 us with both products on the matrix cores, most of it
// those 4 GiB.  Here a wave owns 32 queries and walks the keys in tiles; per
// tile it computes S^T = K Q^T, the running row maximum m, p = exp(s - m),
// and adds V^T P^T to its output, rescaling output and row sum whenever the
// maximum grows, and divides by the sum at the end.
//
// Both products run on the bf16 MFMA over fp32 values split into three bf16
// values (see emit_gemm_split.cpp for the split, its error and its limits).
// The transposed products put a query in a lane: the 32 x 32 x 16 MFMA gives
// lane l the scores of query l % 32 for keys 8 g + 4 (l / 32) + (0 .. 3), and
// wants the same lane's eight values per 16 keys as its operand of the second
// product.  The order of keys inside a product is free, so the tile of V is
// stored in the order the lane already holds and P never leaves its
// registers; a row's maximum and sum need one exchange between the lane's
// two halves of the wave.
//
// Few queries leave most of the chip idle that way: there the waves of a
// workgroup split the keys of one block of 32 queries (see key_split), and
// where even that leaves most of it idle the unfused program is the faster
// one (see attention_pays).
//
// An iteration computes the products of the next tile, the weights of this
// one and the sums of the one before: independent of each other, so that a
// wave's MFMAs run beside its exps and splits (up to six vector instructions
// fit beside one 32-cycle MFMA).
//
// What bounds it: the bf16 MFMAs at the rate the card sustains.  2 x 8 heads
// of 4096 positions, dim 64: 342 us and 8 us for the permute behind it (1438
// us unfused on fp32 MFMAs, 1186 with both products on bf16 ones); the six
// products of the split make that 1.2 PFLOP/s of bf16, against the 1.34-1.42
// that this card's large bf16 products reach.
//
// Accuracy: a weight is exp2((s - m) log2 e) with m the running maximum of s,
// so that a row's largest weight is 1 whatever its scores' size.  (One
// instruction a score less, exp2(fma(s, log2 e, -M)) with M = m log2 e
// rounded, leaves M's rounding in every weight: from scores of 2^31 on the
// largest weight of a row can be 2^-128, where the split keeps four bits.)
// Weights reach the second product in 24 bits relative to the row's maximum
// down to 2^-109 of it; smaller ones lose at most 2^-133, and those below
// 2^-126, which the hardware's exp2 makes zero, all.  With values of V below
// 2^30 that moves an output by at most 2^-96 a key.
// Against 64 bits, normal q, k and v: 1.0e-6 (the unfused program: 1.2e-6).
// What this cannot hold (values of 2^30 and more, infinities and NaN in any
// operand, nonzero Q or K below 2^-109, nonzero V below 2^-109 beside an
// output below 2^-56, sums that are not finite, rows whose scores are all
// -inf) sends the workgroup to `redo`: fp32 MFMAs, in the unfused program's
// order.  The operands are what is looked at, not the scores: below 2^30 no
// product over 128 dims leaves fp32's range, and a NaN that a larger value
// makes in the split need not outlive f (a maximum or minimum of NaN and a
// number is the number).

#include "emit_gemm.hpp"

#include <algorithm>
#include <stdexcept>

namespace porch::cg {

    namespace {

        // A tile of K (rows: keys) or V^T (rows: dims) and how it is read:
        // along its inner side (k: dims of K, keys of V), 128 bits of a row;
        // along its rows, four loads of two rows; or value by value.
        enum class reading { along_k, along_rows, strided };

        struct tile_operand {
            std::string x;      // "K" or "V"
            bool keys_in_rows;  // K: rows are keys; V: the inner side is
            int rows, inner;
            int64_t stride_row, stride_k;
            reading how;
            int units, values;
        };

        tile_operand tile_of(const std::string& x, bool keys_in_rows, int rows, int inner, int64_t stride_row,
                             int64_t stride_k, int threads) {
            tile_operand o{x, keys_in_rows, rows, inner, stride_row, stride_k, reading::strided, 0, 4};
            if (stride_k == 1) o.how = reading::along_k;
            else if (stride_row == 1) o.how = reading::along_rows;
            o.values = o.how == reading::along_rows && rows * inner / 8 >= threads ? 8 : 4;
            o.units = rows * inner / o.values / threads;
            return o;
        }

        // LDS holds [slice of 16][octet][row][h, m, l of 8 values], 48 bytes a
        // row.  Rows of octet o sit at row ^ x(o), so that the octets of a row
        // that adjacent lanes write meet different banks.
        int swizzle_of(const tile_operand& o) { return 128 / o.inner; }

        std::string setup_code(const tile_operand& o, int threads, const char* offset_type) {
            std::string s;
            const std::string OT = offset_type, R = std::to_string(o.rows), X = std::to_string(swizzle_of(o));
            for (int i = 0; i < o.units; ++i) {
                const std::string id = o.x + std::to_string(i);
                s += "    const int c" + id + " = tid + " + std::to_string(i * threads) + ";\n";
                std::string row;
                if (o.how == reading::along_rows) {
                    // adjacent lanes write adjacent LDS rows
                    const std::string across = std::to_string(o.rows * 4 / o.values);
                    s += "    const int oct" + id + " = (c" + id + " >> 1) / " + across + ";\n";
                    s += "    const int half" + id + " = c" + id + " & 1;\n";
                    const std::string at = "((c" + id + " >> 1) % " + across + ")";
                    s += "    const int i" + id + " = " +
                         (o.values == 8 ? at + " * 2" : o.keys_in_rows ? at : "porch_row_dim(" + at + ")") + ";\n";
                    // V's key order: octet h holds keys 4 h .. and 8 + 4 h ..
                    s += "    const int kq" + id + " = " +
                         (o.keys_in_rows ? "oct" + id + " * 8 + half" + id + " * 4"
                                         : "(oct" + id + " >> 1) * 16 + half" + id + " * 8 + (oct" + id + " & 1) * 4") +
                         ";\n";
                }
                else {
                    const std::string per_row = std::to_string(o.inner / 4);
                    s += "    const int kq" + id + " = (c" + id + " % " + per_row + ") * 4;\n";
                    s += "    const int i" + id + " = c" + id + " / " + per_row + ";\n";
                    s += "    const int oct" + id + " = " +
                         (o.keys_in_rows ? "kq" + id + " >> 3"
                                         : "(kq" + id + " >> 4) * 2 + ((kq" + id + " >> 2) & 1)") +
                         ";\n";
                    s += "    const int half" + id + " = (kq" + id + " >> " + (o.keys_in_rows ? "2" : "3") + ") & 1;\n";
                }
                s += "    const " + OT + " o" + id + " = ((" + OT + ")i" + id + " * " + std::to_string(o.stride_row) + " + (" +
                     OT + ")kq" + id + " * " + std::to_string(o.stride_k) + ") * 4;\n";
                for (int e = 0; e < o.values / 4; ++e) {
                    const std::string at = "(i" + id + " + " + std::to_string(e) + ")";
                    s += "    const int w" + id + (e ? "b" : "") + " = (oct" + id + " * " + R + " + (" +
                         (o.keys_in_rows ? at : "porch_dim_row" + at) + " ^ (oct" + id + " * " + X + "))) * 12 + half" +
                         id + " * 2;\n";
                }
            }
            s += "    float r" + o.x + "[" + std::to_string(o.units * o.values) + "];\n";
            return s;
        }

        // The tile whose first key is `key0` into registers; `valid` (empty:
        // all): only keys below it exist, the rest read as zero.
        std::string load_code(const tile_operand& o, const std::string& key0, const std::string& valid,
                              const std::string& ind) {
            const std::string stride = std::to_string(o.keys_in_rows ? o.stride_row : o.stride_k);
            std::string s = ind + "{\n" + ind + "    const char* __restrict__ base = (const char*)(" + o.x + " + (idx_t)(" +
                            key0 + ") * " + stride + ");\n";
            for (int i = 0; i < o.units; ++i) {
                const std::string id = o.x + std::to_string(i);
                auto reg = [&](int j) { return "r" + o.x + "[" + std::to_string(i * o.values + j) + "]"; };
                if (o.how == reading::along_k && (valid.empty() || o.keys_in_rows)) {
                    s += ind + "    porch_f4u v" + id + " = {0.0f, 0.0f, 0.0f, 0.0f};\n";
                    s += ind + "    " + (valid.empty() ? std::string() : "if (i" + id + " < " + valid + ") ") + "v" + id +
                         " = *(const porch_f4u*)(base + o" + id + ");\n" + ind + "    ";
                    const char* e[] = {"x", "y", "z", "w"};
                    for (int j = 0; j < 4; ++j) s += reg(j) + " = v" + id + "." + e[j] + "; ";
                    s += "\n";
                    continue;
                }
                for (int j = 0; j < 4; ++j) {
                    const std::string J = std::to_string(j);
                    const std::string p = "base + o" + id + " + " + std::to_string(j * o.stride_k * 4) + "LL";
                    if (o.values == 8 && (valid.empty() || !o.keys_in_rows)) {
                        s += ind + "    porch_f2u v" + id + J + " = {0.0f, 0.0f};\n";
                        s += ind + "    " + (valid.empty() ? std::string() : "if (kq" + id + " + " + J + " < " + valid + ") ") +
                             "v" + id + J + " = *(const porch_f2u*)(" + p + ");\n";
                        s += ind + "    " + reg(j) + " = v" + id + J + ".x; " + reg(4 + j) + " = v" + id + J + ".y;\n";
                        continue;
                    }
                    for (int e = 0; e < o.values / 4; ++e) {
                        const std::string key = o.keys_in_rows ? "i" + id + " + " + std::to_string(e) : "kq" + id + " + " + J;
                        s += ind + "    " + reg(4 * e + j) + " = " + (valid.empty() ? std::string() : key + " < " + valid + " ? ") +
                             "*(const float*)(" + p + " + " + std::to_string(e * 4) + ")" + (valid.empty() ? "" : " : 0.0f") +
                             ";\n";
                    }
                }
            }
            return s + ind + "}\n";
        }

        std::string store_code(const tile_operand& o, const std::string& buffer, const std::string& ind) {
            std::string s;
            for (int i = 0; i < o.units; ++i)
                for (int e = 0; e < o.values / 4; ++e) {
                    s += ind + "porch_split4(";
                    for (int j = 0; j < 4; ++j) s += "r" + o.x + "[" + std::to_string(i * o.values + 4 * e + j) + "], ";
                    s += "&" + o.x + "s[" + buffer + "][0][0][0] + w" + o.x + std::to_string(i) + (e ? "b" : "") + ", lowest" +
                         o.x + ", largest);\n";
                }
            return s;
        }

        // Can four scores of adjacent keys be emitted together: every input
        // of f at an affine index, no branches.
        bool vector_scores(const kexpr& k, int root) {
            for (const int id : k.postorder(root)) {
                const knode& n = k.at(id);
                if (n.op == kop::select) return false;
                if (n.op == kop::load && !n.index.is_affine) return false;
            }
            return true;
        }

        const char* helpers() {
            return R"(typedef unsigned porch_u4 __attribute__((ext_vector_type(4)));
// LDS row of dim d of V^T: pairs of adjacent dims lie 16 apart.
__device__ __forceinline__ int porch_dim_row(int d) { return (d & ~31) | ((d & 1) << 4) | ((d >> 1) & 15); }
__device__ __forceinline__ int porch_row_dim(int p) { return (p & ~31) | ((p & 15) << 1) | ((p >> 4) & 1); }
)";
        }

        // Two ways to share out the work.  Shared tiles: a workgroup walks all
        // keys for 128 or 256 queries, its waves share each tile of K and V.
        // Split keys: a workgroup takes a block of 32 queries, its waves share
        // out the keys; each wave splits its own K and V into bf16 values, twice
        // the vector work.  Times in us from the rounds of workgroups over the
        // compute units and the tiles of 32 keys that a wave walks, per tile as
        // measured (aligned, one stride over the batch; shared / split / the
        // unfused program): dim 64, 1 x 1024 queries over 1024 keys 67 / 23 /
        // 23, 16 x 2048 over 4096 275 / 290 / 570, 512 x 64 over 4096 662 / 355 /
        // 937; dim 32, 4096 x 32 over 2048 1710 / 473 / 1539; dim 128, 40 x 300
        // over 4096 363 / 273 / 332, 512 x 64 over 32 24.7 / 41 / 21.3.
        struct shares {
            int waves;
            double us;
        };

        int64_t rounds_of(int64_t workgroups, int64_t resident) {
            return (workgroups + resident - 1) / resident;
        }

        shares shared_tiles(int64_t batch, int64_t rows, int64_t keys, int64_t dim, int compute_units) {
            const int64_t cus = std::max(compute_units, 8);
            // Eight waves share each tile of K and V; four where that still
            // leaves no compute unit a second workgroup.
            const int waves = batch * ((rows + 127) / 128) <= cus ? 4 : 8;
            const int64_t rounds = rounds_of(batch * ((rows + 32 * waves - 1) / (32 * waves)), cus);
            const double tile = waves == 4 ? (dim == 32 ? 0.93 : dim == 64 ? 2.05 : 2.8) : (dim == 32 ? 1.65 : dim == 64 ? 2.35 : 6.0);
            return {waves, 4.0 + static_cast<double>(rounds) * (1.5 + static_cast<double>((keys + 31) / 32) * tile)};
        }

        shares split_keys(int64_t batch, int64_t rows, int64_t keys, int64_t dim, int compute_units) {
            const int64_t cus = std::max(compute_units, 8);
            // (four waves fill a compute unit's registers at dim 128, half of
            // them below)
            const int waves = dim == 128 || keys <= 128 ? 4 : 8;
            const int64_t rounds = rounds_of(batch * ((rows + 31) / 32), waves == 4 && dim < 128 ? 2 * cus : cus);
            const int64_t tiles = ((keys + 31) / 32 + waves - 1) / waves;
            const double tile = rounds == 1 ? (dim == 32 ? 2.2 : dim == 64 ? 3.7 : 4.0) : (dim == 32 ? 3.0 : dim == 64 ? 5.0 : 5.2);
            const double fixed = dim == 128 ? 3.5 : (dim == 32 ? 0.5 : 1.5) + (waves == 8 ? dim == 32 ? 1.0 : 1.5 : 0.0);
            return {waves, 4.0 + static_cast<double>(rounds) * (fixed + static_cast<double>(tiles) * tile)};
        }

        // Waves among which the keys of a block of 32 queries are split; 0:
        // none, shared tiles.  Up to two rounds of blocks (one at dim 128) keys
        // are split; past that only entries of few rows, which leave most of a
        // workgroup's waves without queries, and where a launch holds the
        // threads.
        int key_split(int64_t batch, int64_t rows, int64_t keys, int64_t dim, int compute_units) {
            const shares split = split_keys(batch, rows, keys, dim, compute_units);
            const int64_t blocks = batch * ((rows + 31) / 32);
            if (blocks >= (int64_t{1} << 26) / split.waves) return 0;
            if (blocks <= (dim == 128 ? 1 : 2) * static_cast<int64_t>(std::max(compute_units, 8))) return split.waves;
            return rows <= 128 && split.us < shared_tiles(batch, rows, keys, dim, compute_units).us ? split.waves : 0;
        }

    } // namespace

    bool attention_fits(int64_t batch, int64_t rows, int64_t keys, int64_t dim, int64_t value_dim) {
        // a launch holds fewer than 2^32 threads: 512 for 256 queries
        if (batch * ((rows + 255) / 256) >= int64_t{1} << 23) return false;
        return dim == value_dim && (dim == 32 || dim == 64 || dim == 128) && rows >= 32 && keys >= 32;
    }

    bool attention_pays(int64_t batch, int64_t rows, int64_t keys, int64_t dim, bool score_reads, int64_t copied,
                        int compute_units) {
        // No form splits the keys of a block of queries over workgroups, so
        // that few queries over many keys run on a few compute units, where
        // the products and the softmax of the unfused program use them all:
        // dim 64, 1 x 32 queries over 16384 keys 241 us fused, 31 unfused; 8 x
        // 256 over 16384 244 / 165; 64 x 32 over 4096 69 / 92.  The unfused
        // program's launches and split products take 14 to 24 us, its
        // scores (four passes over memory, and matrix cores that a tile of
        // few rows leaves idle) 3.5 to 10.5 us a million, and each operand
        // it can't read in place a copy; a mask costs the kernel a fifth more (its
        // rows are far apart) and the unfused program next to nothing.  That
        // is taken where it is ahead by more than such an estimate is
        // wrong by, up to 1 GiB of scores, for few queries from 1024 keys on
        // (below, both take 20 to 30 us; at dim 128 past 512, from where on
        // the second product is split along K) and for many entries of few rows;
        // with about as many queries as keys and half the compute units at
        // work the kernel's smaller error is worth more than the time (8
        // heads of 1100, dim 128: 4.0e-7 against 4.8e-7, 94 us against 81).
        const int64_t cus = std::max(compute_units, 8), blocks = batch * ((rows + 31) / 32);
        const bool few = keys >= 1024 ? 2 * blocks < cus || keys >= 2 * rows : dim == 128 && keys > 512 && keys >= 2 * rows;
        const bool short_rows = rows < 64 && blocks >= cus;
        if (batch * rows > (int64_t{1} << 28) / keys || !(few || short_rows)) return true;
        const shares form = key_split(batch, rows, keys, dim, compute_units) > 0
                                ? split_keys(batch, rows, keys, dim, compute_units)
                                : shared_tiles(batch, rows, keys, dim, compute_units);
        const double fused = form.us * (score_reads ? 1.2 : 1.0);
        const double launches = dim == 32 ? 14.5 : dim == 64 ? 18.0 : 20.0;
        const double score = rows < 100 ? (dim == 32 ? 4.3 : dim == 64 ? 8.5 : 10.5) : (dim == 32 ? 3.5 : dim == 64 ? 4.3 : 5.2);
        const double unfused = launches + static_cast<double>(batch * rows) * static_cast<double>(keys) * score * 1e-6 +
                               static_cast<double>(copied) * 8.0 / 4e6;
        return fused <= 1.08 * unfused;
    }

    kernel_code emit_attention(const attention_request& r) {
        if (!attention_fits(r.batch, r.rows, r.keys, r.dim, r.dim)) throw std::logic_error("emit_attention: shape");
        const int D = static_cast<int>(r.dim);
        const int split = key_split(r.batch, r.rows, r.keys, r.dim, r.compute_units);
        // keys a tile: two buffers of K and V in 48 KB of LDS (96 at dim 128)
        const int KT = split > 0 ? 32 : std::max(32, 2048 / D);
        const int KB = KT / 32, DB = D / 32, DS = D / 16;
        const bool apart = D == 32; // see gather
        const int waves = split > 0 ? split : shared_tiles(r.batch, r.rows, r.keys, r.dim, r.compute_units).waves;
        const int threads = 64 * waves;
        const int BQ = split > 0 ? 32 : 32 * waves;
        const int64_t tiles = (r.rows + BQ - 1) / BQ;
        const int64_t total = tiles * r.batch;
        const int64_t full = r.keys / KT, tail = r.keys % KT;
        const int64_t steps = full + (tail != 0 ? 1 : 0);
        const std::string SQ = std::to_string(r.rows), SK = std::to_string(r.keys), DD = std::to_string(D);
        const std::string KTS = std::to_string(KT), KBS = std::to_string(KB), DBS = std::to_string(DB), DSS = std::to_string(DS);
        const char* OT = r.width.wide ? "long long" : "unsigned";
        const tile_operand K = tile_of("K", true, KT, D, r.k.stride_col, r.k.stride_row, threads);
        const tile_operand V = tile_of("V", false, D, KT, r.v.stride_col, r.v.stride_row, threads);

        kernel_code kc;
        kc.kind = "attention";
        kc.name = "porch_attention";
        kc.n_slots = r.n_slots;
        kc.block = static_cast<unsigned>(threads);
        kc.grid_x = static_cast<unsigned>(total);
        std::string& s = kc.source;
        s = kernel_prologue(r.n_slots, r.width.type());
        s += bf16_split_helpers();
        s += helpers();
        s += "extern \"C\" __global__ void __launch_bounds__(" + std::to_string(threads) + ", " + (waves == 8 ? "2" : "1") +
             ") porch_attention(" + kernel_params(r.n_slots) + ") {\n";
        if (split > 0) {
            s += "    __shared__ float parts[" + std::to_string(waves) + "][" + std::to_string(16 * DB) + "][64];\n";
            s += "    __shared__ float maxima[" + std::to_string(waves) + "][32], sums[" + std::to_string(waves) + "][32];\n";
        }
        else {
            s += "    __shared__ __attribute__((aligned(16))) float Ks[2][" + DSS + "][" + std::to_string(2 * KT) + "][12];\n";
            s += "    __shared__ __attribute__((aligned(16))) float Vs[2][" + std::to_string(KT / 16) + "][" +
                 std::to_string(2 * D) + "][12];\n";
        }
        s += "    __shared__ unsigned seen[8];\n";
        s += "    const int tid = threadIdx.x;\n    const int lane = tid & 63;\n    const int wave = tid >> 6;\n";
        s += "    const int h = lane >> 5;\n";
        // an XCD takes whole heads where it can: its L2 holds their K and V
        const int64_t each = total / 8, more = total % 8;
        s += "    const int xcd = blockIdx.x % 8;\n";
        s += "    const idx_t lin = (idx_t)xcd * " + std::to_string(each) +
             (more ? " + (xcd < " + std::to_string(more) + " ? xcd : " + std::to_string(more) + ")" : std::string()) +
             " + blockIdx.x / 8;\n";
        if (r.batched) s += "    const idx_t qb = lin / " + std::to_string(tiles) + ";\n";
        s += "    const idx_t own = (lin" + (r.batched ? " % " + std::to_string(tiles) : std::string()) + ") * " +
             std::to_string(BQ) + (split > 0 ? "" : " + wave * 32") + " + (lane & 31);\n";
        s += "    const idx_t q0 = own < " + SQ + " ? own : (idx_t)" + SQ + " - 1;\n";
        auto base = [&](const char* x, const gemm_operand& op) {
            s += std::string("    const float* __restrict__ ") + x + " = a" + std::to_string(op.slot) + " + " +
                 std::to_string(op.offset);
            if (r.batched && op.batch_inner > 0)
                s += " + qb / " + std::to_string(op.batch_inner) + " * " + std::to_string(op.stride_batch_outer) +
                     " + qb % " + std::to_string(op.batch_inner) + " * " + std::to_string(op.stride_batch);
            else if (r.batched && op.stride_batch != 0)
                s += " + qb * " + std::to_string(op.stride_batch);
            s += ";\n";
        };
        base("Q", r.q);
        base("K", r.k);
        base("V", r.v);
        if (split == 0) s += setup_code(K, threads, OT) + setup_code(V, threads, OT);
        s += "    unsigned lowestK = 0xffffffffu, lowestV = 0xffffffffu;\n    porch_s2 largest = {0, 0};\n";
        const std::string partial = std::to_string(full * KT);
        const std::string ahead_of = tail != 0 ? " - 1" : "";
        auto whole = [&](const std::string& g) { return "(" + g + ahead_of + ") * " + KTS; };
        // the partial tile first, so that the loop's loads need no tests
        const std::string valid = tail != 0 ? std::to_string(tail) : "";
        if (split == 0)
            s += load_code(K, tail != 0 ? partial : "0", valid, "    ") + load_code(V, tail != 0 ? partial : "0", valid, "    ");
        // this lane's query, split
        s += "    porch_b8 qf[" + DSS + "][3];\n";
        s += "    #pragma unroll\n    for (int t = 0; t < " + DSS + "; ++t) {\n        porch_u4 u[3];\n";
        s += "        #pragma unroll\n        for (int e = 0; e < 4; ++e) {\n";
        s += "            const idx_t at = q0 * " + std::to_string(r.q.stride_row) + " + (idx_t)(t * 16 + h * 8 + 2 * e) * " +
             std::to_string(r.q.stride_col) + ";\n            unsigned x, y, z;\n";
        s += "            porch_split2(Q[at], Q[at + " + std::to_string(r.q.stride_col) + "], x, y, z, lowestK, largest);\n";
        s += "            u[0][e] = x; u[1][e] = y; u[2][e] = z;\n        }\n";
        s += "        #pragma unroll\n        for (int p = 0; p < 3; ++p) qf[t][p] = __builtin_bit_cast(porch_b8, u[p]);\n    }\n";
        if (split == 0) s += store_code(K, "0", "    ");
        if (split == 0 && steps > 1) {
            s += load_code(K, whole("1"), "", "    ") + store_code(K, "1", "    ");
            s += load_code(K, whole(steps > 2 ? "2" : "1"), "", "    ");
        }
        s += "    float m = -PORCH_FLT_MAX, sum = 0.0f, al = 1.0f;\n    (void)al;\n    porch_v16f acc[" + DBS + "], sc[" + KBS + "];\n    porch_b8 pf[" + std::to_string(KT / 16) + "][3];\n";
        const std::string zero_acc = "    #pragma unroll\n    for (int d = 0; d < " + DBS +
                                     "; ++d)\n        #pragma unroll\n        for (int v = 0; v < 16; ++v) acc[d][v] = 0.0f;\n";
        s += zero_acc;
        if (split == 0) s += "    __syncthreads();\n";

        // f of the 16 products sc[kb][..] of keys key0 + kb 32 + 8 g + 4 h + j
        const bool vec = vector_scores(*r.score_expr, r.score);
        bool score_loads = false;
        for (const int id : r.score_expr->postorder(r.score)) score_loads |= r.score_expr->at(id).op == kop::load;
        auto scores = [&](const std::string& sc, const std::string& key, bool masked, const std::string& ind) {
            std::string c = ind + "#pragma unroll\n" + ind + "for (int g = 0; g < 4; ++g) {\n";
            c += ind + "    const idx_t key = " + key + " + 8 * g + 4 * h;\n" + ind + "    (void)key;\n";
            auto names = [&](const std::string& q1) {
                return r.batched ? std::vector<std::string>{"qb", "q0", q1} : std::vector<std::string>{"q0", q1};
            };
            if (vec && !masked) {
                std::string body;
                emitter em(*r.score_expr, body, 4);
                em.indent = ind + "    ";
                em.declare_roots({r.score});
                em.load = [&](int id) {
                    const knode& n = r.score_expr->at(id);
                    const std::string at = "a" + std::to_string(n.slot);
                    const int64_t w = n.index.w.back();
                    const std::string ix = index_text(n.index, names("key"));
                    if (w == 0) return std::vector<std::string>(4, at + "[" + ix + "]");
                    if (w == 1) {
                        const std::string f = em.fresh("f");
                        em.line("const porch_f4u " + f + " = *(const porch_f4u*)&" + at + "[" + ix + "];");
                        return std::vector<std::string>{f + ".x", f + ".y", f + ".z", f + ".w"};
                    }
                    std::vector<std::string> v;
                    for (int j = 0; j < 4; ++j) v.push_back(at + "[" + ix + " + " + std::to_string(j * w) + "]");
                    return v;
                };
                em.row_value = [](int) { return std::string("porch_lane_product"); };
                em.override_node = [&](int id) {
                    if (r.score_expr->at(id).op != kop::row_value) return std::vector<std::string>{};
                    std::vector<std::string> v;
                    for (int j = 0; j < 4; ++j) v.push_back(sc + "[4 * g + " + std::to_string(j) + "]");
                    return v;
                };
                const std::vector<std::string> v = em.emit(r.score);
                c += body;
                for (int j = 0; j < 4; ++j) c += ind + "    const float x" + std::to_string(j) + " = " + v[static_cast<size_t>(j)] + ";\n";
                for (int j = 0; j < 4; ++j) c += ind + "    " + sc + "[4 * g + " + std::to_string(j) + "] = x" + std::to_string(j) + ";\n";
            }
            else {
                gemm_request e;
                e.expr = r.score_expr;
                e.epilogue = r.score;
                c += ind + "    #pragma unroll\n" + ind + "    for (int j = 0; j < 4; ++j) {\n";
                c += ind + "        const idx_t q1 = key + j" + (masked ? " < " + SK + " ? key + j : (idx_t)" + SK + " - 1" : std::string()) + ";\n";
                c += ind + "        (void)q1;\n" + ind + "        const float acc_v = " + sc + "[4 * g + j];\n";
                std::string body;
                emitter em(*r.score_expr, body, 1);
                em.indent = ind + "        ";
                em.declare_roots({r.score});
                epilogue_emitter(em, e, names("q1"), "acc_v");
                const std::string v = em.emit(r.score)[0];
                c += body + ind + "        " + sc + "[4 * g + j] = " +
                     (masked ? "key + j < " + SK + " ? " + v + " : -__builtin_inff()" : v) + ";\n" + ind + "    }\n";
            }
            return c + ind + "}\n";
        };

        // One wave a SIMD hides its own latencies: an MFMA, an LDS read,
        // six vector instructions, and so on (8 heads of 4096 positions,
        // dim 64: 203 us, five instructions 262).  With two
        // waves a SIMD, or the longer products of dim 128, the compiler's
        // order is the faster one (16 heads of 4096: 365 us against 392).
        auto schedule = [&](const std::string& ind) {
            std::string c;
            if (waves != 4 || D == 128) return c;
            c += ind + "__builtin_amdgcn_sched_group_barrier(0x100, 3, 0);\n";
            for (int i = 0; i < 6 * DS * KB + 6 * (KT / 16) * DB; ++i) {
                c += ind + "__builtin_amdgcn_sched_group_barrier(0x008, 1, 0);\n";
                c += ind + "__builtin_amdgcn_sched_group_barrier(0x100, 1, 0);\n";
                c += ind + "__builtin_amdgcn_sched_group_barrier(0x002, 6, 0);\n";
            }
            return c;
        };
        constexpr int pairs[6][2] = {{0, 0}, {1, 0}, {0, 1}, {1, 1}, {2, 0}, {0, 2}};
        // S^T of one tile of keys from K's buffer `kb` into `sc`
        auto products = [&](const std::string& sc, const std::string& kb, const std::string& ind) {
            std::string c;
            c += ind + "#pragma unroll\n" + ind + "for (int b = 0; b < " + KBS + "; ++b)\n" + ind +
                 "    #pragma unroll\n" + ind + "    for (int v = 0; v < 16; ++v) " + sc + "[b][v] = 0.0f;\n";
            c += ind + "#pragma unroll\n" + ind + "for (int t = 0; t < " + DSS + "; ++t) {\n";
            c += ind + "    const int row = (lane & 31) ^ ((2 * t + h) * " + std::to_string(swizzle_of(K)) + ");\n";
            c += ind + "    porch_b8 kf[" + KBS + "][3];\n";
            c += ind + "    #pragma unroll\n" + ind + "    for (int b = 0; b < " + KBS + "; ++b)\n" + ind + "        #pragma unroll\n" +
                 ind + "        for (int p = 0; p < 3; ++p) kf[b][p] = *(const porch_b8*)&Ks[" + kb + "][t][h * " + KTS +
                 " + b * 32 + row][p * 4];\n";
            for (const auto& pr : pairs)
                c += ind + "    #pragma unroll\n" + ind + "    for (int b = 0; b < " + KBS + "; ++b) " + sc +
                     "[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[b][" + std::to_string(pr[0]) + "], qf[t][" +
                     std::to_string(pr[1]) + "], " + sc + "[b], 0, 0, 0);\n";
            return c + ind + "}\n";
        };
        // the weights of the tile of scores in sc, split into pf, with the
        // new maximum, the sum and the factor `alpha` for what came before
        auto weights = [&](const std::string& key0, bool masked, const std::string& pf, const std::string& ind) {
            std::string c;
            // f's own loads behind the products: 48 heads of 1000 queries over
            // 1023 keys with a mask 66 us against 90
            if (split == 0 && D == 32 && waves == 8 && score_loads) c += ind + "__builtin_amdgcn_sched_barrier(0);\n";
            c += ind + "#pragma unroll\n" + ind + "for (int b = 0; b < " + KBS + "; ++b) {\n";
            c += scores("sc[b]", "(idx_t)(" + key0 + ") + b * 32", masked, ind + "    ");
            c += ind + "}\n";
            // (see `own_tile`; shared tiles of dim 128 in eight waves, loads
            // excepted: 32 heads of 1536 positions 225 us against 244)
            if (split > 0 && D == 32) c += ind + "__builtin_amdgcn_sched_barrier(0);\n";
            if (split == 0 && D == 128 && waves == 8) c += ind + "__builtin_amdgcn_sched_barrier(0x30);\n";
            c += ind + "float tm = sc[0][0];\n";
            c += ind + "#pragma unroll\n" + ind + "for (int b = 0; b < " + KBS + "; ++b)\n" + ind + "    #pragma unroll\n" + ind +
                 "    for (int v = 0; v < 16; ++v) tm = __builtin_fmaxf(tm, sc[b][v]);\n";
            c += ind + "tm = __builtin_fmaxf(tm, __shfl_xor(tm, 32, 64));\n";
            c += ind + "const float mn = __builtin_fmaxf(m, tm);\n";
            c += ind + "const float alpha = __builtin_amdgcn_exp2f((m - mn) * 0x1.715476p+0f);\n" + ind + "m = mn;\n";
            c += ind + "float part[4] = {0.0f, 0.0f, 0.0f, 0.0f};\n";
            c += ind + "#pragma unroll\n" + ind + "for (int b = 0; b < " + KBS + "; ++b)\n" + ind + "    #pragma unroll\n" + ind +
                 "    for (int v = 0; v < 16; ++v) {\n" + ind + "        sc[b][v] = __builtin_amdgcn_exp2f((sc[b][v] - m) * 0x1.715476p+0f);\n" + ind +
                 "        part[v & 3] += sc[b][v];\n" + ind + "    }\n";
            c += ind + "sum = sum * alpha + ((part[0] + part[1]) + (part[2] + part[3]));\n";
            c += ind + "#pragma unroll\n" + ind + "for (int t = 0; t < " + std::to_string(KT / 16) + "; ++t) {\n";
            c += ind + "    porch_u4 u[3];\n" + ind + "    #pragma unroll\n" + ind + "    for (int e = 0; e < 4; ++e) {\n" + ind +
                 "        unsigned x, y, z;\n" + ind +
                 "        porch_split2(sc[t >> 1][(t & 1) * 8 + 2 * e], sc[t >> 1][(t & 1) * 8 + 2 * e + 1], x, y, z);\n" + ind +
                 "        u[0][e] = x; u[1][e] = y; u[2][e] = z;\n" + ind + "    }\n";
            c += ind + "    #pragma unroll\n" + ind + "    for (int p = 0; p < 3; ++p) " + pf +
                 "[t][p] = __builtin_bit_cast(porch_b8, u[p]);\n" + ind + "}\n";
            return c;
        };
        // V^T P^T for the weights in pf and V's buffer `vb`, onto the output.
        // At dim 32 a tile's product is summed by itself, in two chains of
        // MFMAs, and added to the output scaled by `al`, the factor of the
        // maximum before: an output has one rounding a tile at its own size,
        // not one per MFMA (24 heads of 2432 positions: error against 64
        // bits 3.1e-7, and 8.0e-7 with the MFMAs on the output, where the
        // unfused program has 5.1e-7; 126 us against 122).
        auto gather = [&](const std::string& vb, const std::string& ind) {
            std::string c;
            const std::string sums = apart ? "tile[t & 1][d]" : "acc[d]";
            if (apart)
                c += ind + "porch_v16f tile[2][" + DBS + "];\n" + ind + "#pragma unroll\n" + ind + "for (int d = 0; d < " + DBS +
                     "; ++d)\n" + ind + "    #pragma unroll\n" + ind +
                     "    for (int v = 0; v < 16; ++v) tile[0][d][v] = tile[1][d][v] = 0.0f;\n";
            c += ind + "#pragma unroll\n" + ind + "for (int t = 0; t < " + std::to_string(KT / 16) + "; ++t) {\n";
            c += ind + "    const int row = (lane & 31) ^ ((2 * t + h) * " + std::to_string(swizzle_of(V)) + ");\n";
            c += ind + "    porch_b8 vf[" + DBS + "][3];\n";
            c += ind + "    #pragma unroll\n" + ind + "    for (int d = 0; d < " + DBS + "; ++d)\n" + ind + "        #pragma unroll\n" +
                 ind + "        for (int p = 0; p < 3; ++p) vf[d][p] = *(const porch_b8*)&Vs[" + vb + "][t][h * " + DD +
                 " + d * 32 + row][p * 4];\n";
            for (const auto& pr : pairs)
                c += ind + "    #pragma unroll\n" + ind + "    for (int d = 0; d < " + DBS + "; ++d) " + sums +
                     " = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[d][" + std::to_string(pr[0]) + "], pf[t][" +
                     std::to_string(pr[1]) + "], " + sums + ", 0, 0, 0);\n";
            c += ind + "}\n";
            if (apart)
                c += ind + "#pragma unroll\n" + ind + "for (int d = 0; d < " + DBS + "; ++d)\n" + ind + "    #pragma unroll\n" + ind +
                     "    for (int v = 0; v < 16; ++v) acc[d][v] = __builtin_fmaf(acc[d][v], al, tile[0][d][v] + tile[1][d][v]);\n";
            return c;
        };
        // Iteration `it`: the products of tile it + 1, the weights of tile it
        // and the sums of tile it - 1 are independent, so that one wave's MFMAs
        // run beside its exps and splits; K is staged two tiles ahead, V
        // with its weights.
        auto iteration = [&](const std::string& key0, bool first, bool masked) {
            std::string c;
            const std::string ind = "        ";
            c += ind + "porch_v16f sn[" + KBS + "];\n" + products("sn", "(it + 1) & 1", ind);
            if (!first) c += gather("(it - 1) & 1", ind);
            c += ind + "porch_b8 pn[" + std::to_string(KT / 16) + "][3];\n";
            c += weights(key0, masked, "pn", ind);
            if (steps > 1) c += store_code(K, "it & 1", ind);
            c += store_code(V, "it & 1", ind);
            if (steps > 1) {
                c += ind + "const int ak = it + 3 < " + std::to_string(steps) + " ? it + 3 : " + std::to_string(steps - 1) + ";\n";
                c += load_code(K, whole("ak"), "", ind);
                c += ind + "const int av = it + 1 < " + std::to_string(steps) + " ? it + 1 : " + std::to_string(steps - 1) + ";\n";
                c += load_code(V, whole("av"), "", ind);
            }
            if (apart) c += ind + "al = alpha;\n";
            else if (!first)
                c += ind + "#pragma unroll\n" + ind + "for (int d = 0; d < " + DBS + "; ++d)\n" + ind + "    #pragma unroll\n" + ind +
                     "    for (int v = 0; v < 16; ++v) acc[d][v] *= alpha;\n";
            c += ind + "#pragma unroll\n" + ind + "for (int b = 0; b < " + KBS + "; ++b) sc[b] = sn[b];\n";
            c += ind + "#pragma unroll\n" + ind + "for (int i = 0; i < " + std::to_string(KT / 16) + "; ++i)\n" + ind +
                 "    #pragma unroll\n" + ind + "    for (int p = 0; p < 3; ++p) pf[i][p] = pn[i][p];\n";
            if (!first) c += schedule(ind);
            c += ind + "__syncthreads();\n";
            return c;
        };
        // Split keys: wave w takes the tiles w, w + waves, .. and reads their
        // fragments from memory as the MFMAs want them (lane: a key of K, a
        // dim of V, eight values along the product); no wave waits for
        // another until the end.
        auto fragments = [&](const std::string& key0, bool masked, const std::string& ind) {
            std::string c;
            const std::string limit = " < " + SK + " ? kx : (idx_t)" + SK + " - 1";
            c += ind + "#pragma unroll\n" + ind + "for (int t = 0; t < " + DSS + "; ++t)\n" + ind + "    #pragma unroll\n" + ind +
                 "    for (int b = 0; b < " + KBS + "; ++b) {\n";
            c += ind + "        const idx_t kx = " + key0 + " + b * 32 + (lane & 31);\n";
            c += ind + "        const float* const at = K + (" + (masked ? "kx" + limit : std::string("kx")) + ") * " +
                 std::to_string(r.k.stride_col) + " + (idx_t)(t * 16 + h * 8) * " + std::to_string(r.k.stride_row) + ";\n";
            if (r.k.stride_row == 1)
                c += ind + "        const porch_f4u x = *(const porch_f4u*)at, y = *(const porch_f4u*)(at + 4);\n" + ind +
                     "        #pragma unroll\n" + ind + "        for (int e = 0; e < 4; ++e) { kr[t][b][e] = x[e]; kr[t][b][4 + e] = y[e]; }\n";
            else
                c += ind + "        #pragma unroll\n" + ind + "        for (int e = 0; e < 8; ++e) kr[t][b][e] = at[(idx_t)e * " +
                     std::to_string(r.k.stride_row) + "];\n";
            c += ind + "    }\n";
            c += ind + "#pragma unroll\n" + ind + "for (int t = 0; t < " + std::to_string(KT / 16) + "; ++t)\n" + ind +
                 "    #pragma unroll\n" + ind + "    for (int d = 0; d < " + DBS + "; ++d) {\n";
            c += ind + "        const float* const at = V + (idx_t)(d * 32 + porch_row_dim(lane & 31)) * " +
                 std::to_string(r.v.stride_col) + ";\n";
            if (r.v.stride_row == 1 && !masked)
                c += ind + "        const porch_f4u x = *(const porch_f4u*)(at + " + key0 + " + t * 16 + 4 * h), y = *(const porch_f4u*)(at + " +
                     key0 + " + t * 16 + 4 * h + 8);\n" + ind +
                     "        #pragma unroll\n" + ind + "        for (int e = 0; e < 4; ++e) { vr[t][d][e] = x[e]; vr[t][d][4 + e] = y[e]; }\n";
            else
                c += ind + "        #pragma unroll\n" + ind + "        for (int e = 0; e < 8; ++e) {\n" + ind +
                     "            const idx_t kx = " + key0 + " + t * 16 + 4 * h + (e & 3) + (e & 4) * 2;\n" + ind +
                     "            vr[t][d][e] = at[(" + (masked ? "kx" + limit : std::string("kx")) + ") * " + std::to_string(r.v.stride_row) +
                     "];\n" + ind + "        }\n";
            return c + ind + "    }\n";
        };
        auto own_tile = [&](bool masked) {
            const std::string ind = "            ";
            std::string c = fragments("key0", masked, ind);
            auto split8 = [&](const std::string& from, const std::string& lowest) {
                return ind + "    porch_b8 f[3];\n" + ind + "    {\n" + ind + "        porch_u4 u[3];\n" + ind +
                       "        #pragma unroll\n" + ind + "        for (int e = 0; e < 4; ++e) {\n" + ind +
                       "            unsigned x, y, z;\n" + ind + "            porch_split2(" + from + "[2 * e], " + from +
                       "[2 * e + 1], x, y, z, " + lowest + ", largest);\n" + ind +
                       "            u[0][e] = x; u[1][e] = y; u[2][e] = z;\n" + ind + "        }\n" + ind +
                       "        #pragma unroll\n" + ind + "        for (int p = 0; p < 3; ++p) f[p] = __builtin_bit_cast(porch_b8, u[p]);\n" +
                       ind + "    }\n";
            };
            c += ind + "#pragma unroll\n" + ind + "for (int b = 0; b < " + KBS + "; ++b)\n" + ind +
                 "    #pragma unroll\n" + ind + "    for (int v = 0; v < 16; ++v) sc[b][v] = 0.0f;\n";
            c += ind + "#pragma unroll\n" + ind + "for (int b = 0; b < " + KBS + "; ++b)\n" + ind + "#pragma unroll\n" + ind +
                 "for (int t = 0; t < " + DSS + "; ++t) {\n" + split8("kr[t][b]", "lowestK");
            for (const auto& pr : pairs)
                c += ind + "    sc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[" + std::to_string(pr[0]) + "], qf[t][" +
                     std::to_string(pr[1]) + "], sc[b], 0, 0, 0);\n";
            c += ind + "}\n";
            // V is split after the weights, and at dim 32 f's own loads come
            // before them: in the compiler's order the weights wait for loads
            // that they have no use for (64 heads of 32 queries over 4099 keys,
            // dim 128 229 us against 149; 16 of 77 over 12288 with a mask, dim
            // 32 162 against 131).
            c += weights("key0", masked, "pf", ind);
            c += ind + "__builtin_amdgcn_sched_barrier(0);\n";
            c += ind + "#pragma unroll\n" + ind + "for (int d = 0; d < " + DBS + "; ++d) {\n";
            c += ind + "    porch_v16f own_sum;\n" + ind + "    #pragma unroll\n" + ind + "    for (int v = 0; v < 16; ++v) own_sum[v] = 0.0f;\n";
            c += ind + "    #pragma unroll\n" + ind + "    for (int t = 0; t < " + std::to_string(KT / 16) + "; ++t) {\n" + split8("vr[t][d]", "lowestV");
            for (const auto& pr : pairs)
                c += ind + "        own_sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[" + std::to_string(pr[0]) + "], pf[t][" +
                     std::to_string(pr[1]) + "], own_sum, 0, 0, 0);\n";
            c += ind + "    }\n";
            c += ind + "    #pragma unroll\n" + ind + "    for (int v = 0; v < 16; ++v) acc[d][v] = __builtin_fmaf(acc[d][v], alpha, own_sum[v]);\n" + ind + "}\n";
            return c;
        };
        if (split > 0) {
            s += "    float kr[" + DSS + "][" + KBS + "][8], vr[" + std::to_string(KT / 16) + "][" + DBS + "][8];\n";
            s += "    for (int it = wave; it < " + std::to_string(steps) + "; it += " + std::to_string(waves) + ") {\n";
            s += "        const idx_t key0 = (idx_t)it * " + KTS + ";\n";
            if (tail == 0) s += "        {\n" + own_tile(false) + "        }\n    }\n";
            else if (full == 0) s += "        {\n" + own_tile(true) + "        }\n    }\n";
            else
                s += "        if (it < " + std::to_string(full) + ") {\n" + own_tile(false) + "        }\n        else {\n" +
                     own_tile(true) + "        }\n    }\n";
        }
        else {
            s += products("sc", "0", "    ") + "    __syncthreads();\n";
            s += "    {\n        const int it = 0;\n" + iteration(tail != 0 ? partial : "0", true, tail != 0) + "    }\n";
            if (steps > 1)
                s += "    for (int it = 1; it < " + std::to_string(steps) + "; ++it) {\n" + iteration(whole("it"), false, false) + "    }\n";
            s += gather(std::to_string((steps - 1) & 1), "    ");
        }

        // what the split could not hold
        s += "    sum += __shfl_xor(sum, 32, 64);\n";
        if (split > 0) {
            // the row's maximum and sum over all waves (a wave whose keys
            // are all masked has a sum of 0)
            s += "    if (lane < 32) {\n        maxima[wave][lane] = m;\n        sums[wave][lane] = sum;\n    }\n    __syncthreads();\n";
            s += "    float row_max = maxima[0][lane & 31], row_sum = 0.0f;\n    #pragma unroll\n    for (int w = 1; w < " +
                 std::to_string(waves) + "; ++w) row_max = __builtin_fmaxf(row_max, maxima[w][lane & 31]);\n";
            s += "    #pragma unroll\n    for (int w = 0; w < " + std::to_string(waves) +
                 "; ++w) row_sum += sums[w][lane & 31] * __builtin_amdgcn_exp2f((maxima[w][lane & 31] - row_max) * 0x1.715476p+0f);\n";
            s += "    float share = __builtin_amdgcn_exp2f((m - row_max) * 0x1.715476p+0f);\n    sum = row_sum;\n";
        }
        s += "    bool wrong = largest.x >= 0x4e80 || largest.y >= 0x4e80 || !(sum > 0.0f && sum <= PORCH_FLT_MAX), small = false;\n";
        s += "    #pragma unroll\n    for (int d = 0; d < " + DBS + "; ++d)\n        #pragma unroll\n        for (int v = 0; v < 16; ++v) {\n";
        s += "            const float x = __builtin_fabsf(acc[d][v]);\n";
        s += "            wrong |= !(x <= PORCH_FLT_MAX);\n            small |= !(x >= 0x1p-56f);\n        }\n";
        s += "    const unsigned found = (__ballot(wrong || lowestK < 0x12000000u) != 0 ? 1u : 0u) |\n"
             "                           (__ballot(small) != 0 ? 2u : 0u) |\n"
             "                           (__ballot(lowestV < 0x12000000u) != 0 ? 4u : 0u);\n";
        s += "    if (lane == 0) seen[wave] = found;\n    __syncthreads();\n";
        s += "    unsigned all = 0;\n    #pragma unroll\n    for (int w = 0; w < " + std::to_string(waves) + "; ++w) all |= seen[w];\n";
        // In fp32 throughout, in the order of the unfused program: every
        // row's maximum and sum first, then the weights, divided before they
        // meet V (undivided, large values could overflow).
        // (Split keys: the first wave, with all of them.)
        s += "    if ((all & 1u) != 0 || (all & 6u) == 6u) {\n" + zero_acc;
        if (split > 0) s += "        share = wave == 0 ? 1.0f : 0.0f;\n        if (wave == 0) {\n";
        s += "        m = -PORCH_FLT_MAX;\n        sum = 0.0f;\n";
        s += "        for (int pass = 0; pass < 2; ++pass) {\n        for (int key0 = 0; key0 < " + SK + "; key0 += 32) {\n";
        s += "            porch_v16f sc;\n            #pragma unroll\n            for (int v = 0; v < 16; ++v) sc[v] = 0.0f;\n";
        s += "            const idx_t kr = key0 + (lane & 31) < " + SK + " ? key0 + (lane & 31) : " + SK + " - 1;\n";
        s += "            for (int d = 0; d < " + DD + "; d += 2)\n";
        s += "                sc = __builtin_amdgcn_mfma_f32_32x32x2f32(K[kr * " + std::to_string(r.k.stride_col) + " + (idx_t)(d + h) * " +
             std::to_string(r.k.stride_row) + "], Q[q0 * " + std::to_string(r.q.stride_row) + " + (idx_t)(d + h) * " +
             std::to_string(r.q.stride_col) + "], sc, 0, 0, 0);\n";
        s += scores("sc", "(idx_t)key0", true, "            ");
        s += "            if (pass == 0) {\n";
        s += "                float tm = sc[0];\n                #pragma unroll\n                for (int v = 0; v < 16; ++v) tm = __builtin_fmaxf(tm, sc[v]);\n";
        s += "                tm = __builtin_fmaxf(tm, __shfl_xor(tm, 32, 64));\n                const float mn = __builtin_fmaxf(m, tm);\n";
        s += "                float part = 0.0f;\n                #pragma unroll\n                for (int v = 0; v < 16; ++v) part += porch_exp(sc[v] - mn);\n";
        s += "                sum = sum * porch_exp(m - mn) + part;\n                m = mn;\n            }\n";
        s += "            else {\n                #pragma unroll\n                for (int v = 0; v < 16; ++v) sc[v] = porch_exp(sc[v] - m) / sum;\n";
        s += "                #pragma unroll\n                for (int d = 0; d < " + DBS + "; ++d)\n                    #pragma unroll\n                    for (int v = 0; v < 16; ++v) {\n";
        s += "                        const int key = key0 + 8 * (v >> 2) + 4 * h + (v & 3);\n";
        s += "                        const float x = key < " + SK + " ? V[(idx_t)key * " + std::to_string(r.v.stride_row) +
             " + (idx_t)porch_row_dim(d * 32 + (lane & 31)) * " + std::to_string(r.v.stride_col) + "] : 0.0f;\n";
        s += "                        acc[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, sc[v], acc[d], 0, 0, 0);\n";
        s += "                    }\n            }\n        }\n";
        s += "        if (pass == 0) sum += __shfl_xor(sum, 32, 64);\n        }\n";
        if (split > 0) s += "        }\n";
        s += "        sum = 1.0f; // divided already\n    }\n";

        // Output: register v of block d holds dim d 32 + 16 (v / 4 % 2) + 8 h +
        // 2 (v % 4) + v / 8: eight adjacent dims a lane from four registers of
        // either half of a block.
        if (split > 0) {
            s += "    #pragma unroll\n    for (int d = 0; d < " + DBS + "; ++d)\n        #pragma unroll\n        for (int v = 0; v < 16; ++v) parts[wave][d * 16 + v][lane] = acc[d][v] * share;\n";
            s += "    __syncthreads();\n";
        }
        s += "    if (own < " + SQ + ") {\n";
        if (split > 0) {
            // the waves share the sums of their parts: 8 values a lane each
            s += "        for (int u = wave; u < " + std::to_string(2 * DB) + "; u += " + std::to_string(waves) + ") {\n";
            s += "            const int d = u >> 1, g = u & 1;\n";
        }
        else
            s += "        #pragma unroll\n        for (int d = 0; d < " + DBS + "; ++d)\n        #pragma unroll\n        for (int g = 0; g < 2; ++g) {\n";
        s += "            float y[8];\n            const idx_t qn = d * 32 + 16 * g + 8 * h;\n";
        s += "            #pragma unroll\n            for (int e = 0; e < 8; ++e) {\n";
        if (split > 0) {
            s += "                const int at = d * 16 + (e & 1) * 8 + 4 * g + (e >> 1);\n                float all_keys = parts[0][at][lane];\n";
            s += "                #pragma unroll\n                for (int w = 1; w < " + std::to_string(waves) + "; ++w) all_keys += parts[w][at][lane];\n";
            s += "                const float acc_v = all_keys / sum;\n";
        }
        else
            s += "                const float acc_v = acc[d][(e & 1) * 8 + 4 * g + (e >> 1)] / sum;\n";
        s += "                const idx_t q1 = qn + e;\n                (void)q1;\n";
        {
            gemm_request e;
            e.expr = r.expr;
            e.epilogue = r.epilogue;
            std::string body;
            emitter em(*r.expr, body, 1);
            em.indent = "                ";
            em.declare_roots({r.epilogue});
            epilogue_emitter(em, e, r.batched ? std::vector<std::string>{"qb", "q0", "q1"} : std::vector<std::string>{"q0", "q1"},
                             "acc_v");
            const std::string v = em.emit(r.epilogue)[0];
            s += body + "                y[e] = " + v + ";\n            }\n";
        }
        s += "            float* const to = out + " + std::string(r.batched ? "(qb * " + SQ + " + q0) * " : "q0 * ") + DD + " + qn;\n";
        s += "            #pragma unroll\n            for (int e = 0; e < 8; e += 4) {\n";
        s += "                porch_f4u z = {y[e], y[e + 1], y[e + 2], y[e + 3]};\n                *(porch_f4u*)(to + e) = z;\n            }\n";
        s += "        }\n    }\n}\n";
        return kc;
    }

} // namespace porch::cg
