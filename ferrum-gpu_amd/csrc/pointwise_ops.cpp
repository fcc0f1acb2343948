// pointwise_ops.cpp -- see pointwise_ops.hpp.
#include "pointwise_ops.hpp"

#include <algorithm>

#include <initializer_list>
#include <string>

#include "kernels/tile_geom.h"

namespace fg {

namespace {

constexpr uint32_t kThreads = 256;
constexpr uint64_t kMaxBlocks = 1u << 16;  // 16.8 M threads; the kernels stride over the rest

bool aligned16(std::initializer_list<const void*> ps) {
    for (const void* p : ps)
        if (reinterpret_cast<uintptr_t>(p) & 15u) return false;
    return true;
}

void need_ptrs(const char* op, std::initializer_list<const void*> ps) {
    for (const void* p : ps)
        if (!p) invalid(std::string(op) + ": null buffer");
}

// Input and output ranges of n complex (8n bytes) or n floats (4n bytes) must
// be identical or disjoint where the kernel reads one array and writes another
// with a different stride.
bool overlap(const void* a, uint64_t abytes, const void* b, uint64_t bbytes) {
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return x < y + bbytes && y < x + abytes;
}

// The kernels' last argument: whether they load their inputs through the
// caches, by the bytes of one complex array of n elements.  From 12 MiB up to
// 40 MiB for a product (which reads two arrays) and 80 MiB for a conversion.
// Below, a launch is bound by the host; above, the inputs no longer fit the
// Infinity Cache beside the output.  Measured on gfx950: us per launch with
// streamed loads and the change, in percent, with cached ones, for the same
// buffers each time, three sets in turn, and buffers last touched 1.2 GB of
// other traffic before ("cold"); the caches are flushed between settings and
// warmed by each setting itself:
//                             the same  in turn    cold
//   product, in place 12 MiB  7.5 -34   8.0 -13    8.1 +12
//                     16 MiB  9.4 -47   9.8 -11    10.0 +14
//                     32 MiB  17.1 -9   17.7 -14   17.6 +11
//   out of place      16 MiB  9.3 -28   9.9 -12    10.1 +3
//                     24 MiB  13.1 -9   13.7 -13   13.9 +3
//                     36 MiB  18.9 -10  19.4 -11   19.4 +4
//                     48 MiB  24.4 -11  25.0 +5    25.0 +5
//   split             24 MiB  13.5 -8   14.7 -15   14.9 +5
//   interleave        12 MiB  6.1 -20   6.4 -19    6.6 +2
//                     24 MiB  10.3 -50  10.7 -16   10.9 +4
//                     79 MiB  28.4 -13  28.6 -15   28.6 +2
//   deinterleave      24 MiB  9.9 -47   10.3 -16   10.3 +5
// (A product over the same 20 to 28 MiB arrays, just written and never
// displaced, runs 3 to 7 % faster streamed.)  The product within a filter
// (transform, product, inverse, in place) gains on multi-launch plans: 1024 x
// 1024 24 MiB 63.9 -5, 62.3 -5, 64.7 -2, 512 x 512 32 MiB 73.0 -10, 72.9 -4,
// 76.1 -8 (12 MiB 45.7 +2, 42.4 +2, 44.0 +2), 2^16 points 24 MiB 58.3 -6, 58.1
// -6, 59.8 -4.  It loses on single-pass plans below about 30 MiB, whose
// outputs were streamed out and are not in the caches: 256 points 23 MiB 30.8
// +7, 30.9 +7, 31.1 +11, 1024 points 16 MiB 24.2 +5, 25.3 +5, 27.5 +5, 35 MiB
// 48.7 -9, 47.0 -2, 52.4 -7.  A product does not know what wrote its inputs;
// the range weighs these.
uint32_t load_flags(uint64_t n, uint64_t limit) {
    const uint64_t mib = n >> 17;  // of 8 n bytes
    return mib >= 12 && mib < limit ? FG_PASS_LOAD_CACHED : 0u;
}
constexpr uint64_t kProductMiB = 40, kConvertMiB = 80;

void launch(const HipBackend::DeviceHandle& dev, hipStream_t stream, HipBackend::KernelHandle k, uint64_t n,
            int width, void** args) {
    const uint64_t chunks = (n + width - 1) / width;
    uint64_t blocks = (chunks + kThreads - 1) / kThreads;
    if (blocks > kMaxBlocks) blocks = kMaxBlocks;
    HipBackend::launch(dev, stream, k, Dim3((uint32_t)blocks), Dim3(kThreads), 0, args);
}

}  // namespace

Pointwise::Pointwise(const HipBackend::Module& mod) {
    for (int v = 0; v < 2; ++v) {
        const std::string w = v ? "_vec" : "_elem";
        cmul_c64_[v] = HipBackend::get_kernel(mod, ("fg_cmul_c64" + w).c_str());
        cmul_split_[v] = HipBackend::get_kernel(mod, ("fg_cmul_split" + w).c_str());
        deinterleave_[v] = HipBackend::get_kernel(mod, ("fg_deinterleave_c64" + w).c_str());
        interleave_[v] = HipBackend::get_kernel(mod, ("fg_interleave_c64" + w).c_str());
    }
    fill_ = HipBackend::get_kernel(mod, "fg_fill_c64");
    transpose_ = HipBackend::get_kernel(mod, "fg_transpose_c64");
    transpose128_ = HipBackend::get_kernel(mod, "fg_transpose_c64_t128");
    copy_ = HipBackend::get_kernel(mod, "fg_copy_f4");
}

void Pointwise::cmul_c64(const HipBackend::DeviceHandle& dev, const void* a, const void* b, void* out, uint64_t n,
                         hipStream_t stream) const {
    if (n == 0) return;
    need_ptrs("cmul_c64", {a, b, out});
    // Element i of out depends only on element i of a and b: out may be a or b,
    // but must not overlap either at another offset.
    for (const void* x : {a, b})
        if (x != out && overlap(out, 8 * n, x, 8 * n)) invalid("cmul_c64: out partially overlaps an input");
    const int v = aligned16({a, b, out}) ? 1 : 0;
    uint32_t flags = load_flags(n, kProductMiB);
    void* args[] = {(void*)&a, (void*)&b, &out, &n, &flags};
    launch(dev, stream, cmul_c64_[v], n, v ? 2 : 1, args);
}

void Pointwise::cmul_split(const HipBackend::DeviceHandle& dev, const void* a_re, const void* a_im,
                           const void* b_re, const void* b_im, void* o_re, void* o_im, uint64_t n,
                           hipStream_t stream) const {
    if (n == 0) return;
    need_ptrs("cmul_split", {a_re, a_im, b_re, b_im, o_re, o_im});
    const uint64_t nb = 4 * n;
    // Element i of the outputs depends only on element i of the inputs, so
    // o_re may be a_re or b_re and o_im may be a_im or b_im; any other overlap
    // of an output with an input or with the other output is rejected.
    for (const void* x : {a_re, b_re, a_im, b_im}) {
        const bool same_part_re = x == a_re || x == b_re;
        if (!(same_part_re && x == o_re) && overlap(o_re, nb, x, nb))
            invalid("cmul_split: o_re overlaps an input other than a_re / b_re");
        if (!(!same_part_re && x == o_im) && overlap(o_im, nb, x, nb))
            invalid("cmul_split: o_im overlaps an input other than a_im / b_im");
    }
    if (overlap(o_re, nb, o_im, nb)) invalid("cmul_split: o_re and o_im overlap");
    const int v = aligned16({a_re, a_im, b_re, b_im, o_re, o_im}) ? 1 : 0;
    uint32_t flags = load_flags(n, kProductMiB);
    void* args[] = {(void*)&a_re, (void*)&a_im, (void*)&b_re, (void*)&b_im, &o_re, &o_im, &n, &flags};
    launch(dev, stream, cmul_split_[v], n, v ? 4 : 1, args);
}

void Pointwise::deinterleave(const HipBackend::DeviceHandle& dev, const void* in, void* re, void* im, uint64_t n,
                             hipStream_t stream) const {
    if (n == 0) return;
    need_ptrs("deinterleave", {in, re, im});
    if (overlap(in, 8 * n, re, 4 * n) || overlap(in, 8 * n, im, 4 * n) || overlap(re, 4 * n, im, 4 * n))
        invalid("deinterleave: buffers overlap");
    const int v = aligned16({in, re, im}) ? 1 : 0;
    uint32_t flags = load_flags(n, kConvertMiB);
    void* args[] = {(void*)&in, &re, &im, &n, &flags};
    launch(dev, stream, deinterleave_[v], n, v ? 2 : 1, args);
}

void Pointwise::interleave(const HipBackend::DeviceHandle& dev, const void* re, const void* im, void* out,
                           uint64_t n, hipStream_t stream) const {
    if (n == 0) return;
    need_ptrs("interleave", {re, im, out});
    if (overlap(out, 8 * n, re, 4 * n) || overlap(out, 8 * n, im, 4 * n)) invalid("interleave: buffers overlap");
    const int v = aligned16({re, im, out}) ? 1 : 0;
    uint32_t flags = load_flags(n, kConvertMiB);
    void* args[] = {(void*)&re, (void*)&im, &out, &n, &flags};
    launch(dev, stream, interleave_[v], n, v ? 2 : 1, args);
}

void Pointwise::fill_c64(const HipBackend::DeviceHandle& dev, void* out, uint64_t n, uint64_t seed, bool normal,
                         hipStream_t stream) const {
    if (n == 0) return;
    need_ptrs("fill_c64", {out});
    if (reinterpret_cast<uintptr_t>(out) & 7u) invalid("fill_c64: out must be 8-byte aligned (complex64)");
    uint32_t nrm = normal ? 1u : 0u;
    void* args[] = {&out, &n, &seed, &nrm};
    launch(dev, stream, fill_, n, 1, args);
}

void Pointwise::transpose_c64(const HipBackend::DeviceHandle& dev, const void* in, void* out, uint32_t rows,
                              uint32_t cols, uint64_t batch, hipStream_t stream) const {
    if (!in || !out) invalid("transpose: null buffer");
    if (rows == 0 || cols == 0 || batch == 0) invalid("transpose: rows, cols and batch must be positive");
    const uint64_t nb = 8ull * rows * cols * batch;
    if (overlap(in, nb, out, nb)) invalid("transpose: in and out must not overlap");
    if (rows >= 128 && cols >= 128) {
        // 128 x 128 tiles walked in super-tiles of up to 8 x 8 (fg_transpose_c64_t128)
        const uint32_t tc = (cols + 127) / 128, tr = (rows + 127) / 128;
        const uint32_t sc = std::min<uint32_t>(8, tc), sr = std::min<uint32_t>(8, tr);
        const uint32_t supers_c = (tc + sc - 1) / sc, supers_r = (tr + sr - 1) / sr;
        const uint64_t image_blocks = (uint64_t)supers_c * sc * supers_r * sr;
        if (image_blocks * batch > 0x7fffffffull) invalid("transpose: too many tiles for one launch");
        uint32_t ib = (uint32_t)image_blocks;
        void* args[] = {(void*)&in, &out, &rows, &cols, (void*)&tc, (void*)&tr, (void*)&sc, (void*)&sr,
                        (void*)&supers_c, &ib};
        HipBackend::launch(dev, stream, transpose128_, Dim3((uint32_t)(image_blocks * batch)), Dim3(1024), 0, args);
        return;
    }
    const uint32_t tc = (cols + 63) / 64, tr = (rows + 63) / 64;
    const uint64_t tiles = (uint64_t)tc * tr * batch;
    if (tiles > 0x7fffffffull) invalid("transpose: too many tiles for one launch");
    void* args[] = {(void*)&in, &out, &rows, &cols, (void*)&tc, (void*)&tr};
    HipBackend::launch(dev, stream, transpose_, Dim3((uint32_t)tiles), Dim3(256), 0, args);
}

void Pointwise::stream_copy(const HipBackend::DeviceHandle& dev, const void* in, void* out, uint64_t bytes,
                            hipStream_t stream) const {
    need_ptrs("stream_copy", {in, out});
    if (bytes % 16) invalid("fg_stream_copy: bytes must be a multiple of 16");
    if (!aligned16({in, out})) invalid("fg_stream_copy: d_in and d_out must be 16-byte aligned");
    uint64_t n4 = bytes / 16;
    const uint32_t block = 64;
    uint64_t blocks = (n4 + block - 1) / block;
    if (blocks > 0x7fffffffull) blocks = 0x7fffffffull;  // the kernel strides beyond this
    if (blocks == 0) return;
    void* args[] = {(void*)&in, &out, &n4};
    HipBackend::launch(dev, stream, copy_, Dim3((uint32_t)blocks), Dim3(block), 0, args);
}

}  // namespace fg
