// C ABI of libfa_mi355.so (declared in include/fa_mi355.h): argument validation and dispatch.
// Host code only; the kernels live in fa_fwd.hip, fa_bwd.hip, fa_bwd_narrow.hip (dK, dV and dBias of the small head dims) and
// fa_bwd_shared.hip (the gradient of a shared bias).
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
#include <mutex>

#include "../../include/fa_mi355.h"
#include "fa_params.hpp"

namespace fa {
// one object file per head dimension defines these (fa_fwd.hip, fa_bwd.hip, fa_bwd_shared.hip with -DFA_HEAD_DIM)
template <int D> hipError_t launch_fwd_d(const FwdParams& p, int dtype, int bias, bool causal, hipStream_t st);
template <int D> hipError_t launch_bwd_d(const BwdParams& p, int dtype, int bias, bool causal, int dbias, int stages, hipStream_t st);
template <int D> hipError_t launch_bwd_shared_d(const BwdParams& p, int dtype, hipStream_t st);
#define FA_DECLARE_D(D)                                                                                         \
    template <> hipError_t launch_fwd_d<D>(const FwdParams& p, int dtype, int bias, bool causal, hipStream_t st); \
    template <> hipError_t launch_bwd_d<D>(const BwdParams& p, int dtype, int bias, bool causal, int dbias, int stages, hipStream_t st);
#define FA_DECLARE_SHARED_D(D) template <> hipError_t launch_bwd_shared_d<D>(const BwdParams& p, int dtype, hipStream_t st);
FA_DECLARE_D(16)
FA_DECLARE_D(32)
FA_DECLARE_D(64)
FA_DECLARE_D(96)
FA_DECLARE_D(128)
FA_DECLARE_D(256)
FA_DECLARE_SHARED_D(16)
FA_DECLARE_SHARED_D(32)
FA_DECLARE_SHARED_D(64)
FA_DECLARE_SHARED_D(128)
FA_DECLARE_SHARED_D(256)
#undef FA_DECLARE_D
#undef FA_DECLARE_SHARED_D

// Head dims of a D = 128 problem that fit 96: three quarters of the products, copies and LDS, and the dK / dV kernel of the
// small head dims where no bias tile is streamed.  Forward / backward, us, at 128 -> at 96: B=2 H=16 M=N=4096 D=96 250 / 829 ->
// 208 / 634, B=16 H=12 S=512 D=72 39.0 / 127 -> 32.1 / 100, ALiBi B=4 H=8 S=1024 D=96 44.6 / 89 -> 37.5 / 80.
static int tight_head_dim(int D, int d_qk, int d_v) { return D == 128 && d_qk <= 96 && d_v <= 96 ? 96 : D; }

static hipError_t launch_fwd(const FwdParams& p, int D, int dtype, int bias, bool causal, hipStream_t st) {
    switch (tight_head_dim(D, p.d_qk, p.d_v)) {
        case 16: return launch_fwd_d<16>(p, dtype, bias, causal, st);
        case 32: return launch_fwd_d<32>(p, dtype, bias, causal, st);
        case 64: return launch_fwd_d<64>(p, dtype, bias, causal, st);
        case 96: return launch_fwd_d<96>(p, dtype, bias, causal, st);
        case 128: return launch_fwd_d<128>(p, dtype, bias, causal, st);
        case 256: return launch_fwd_d<256>(p, dtype, bias, causal, st);
    }
    return hipErrorNotSupported;
}
static hipError_t launch_bwd(const BwdParams& p, int D, int dtype, int bias, bool causal, int dbias, int stages, hipStream_t st) {
    const bool bias_tile = bias >= 1 && bias <= 4 && !(p.row_bias_kind != 0 && dbias != 1);
    const int kernel_dim = bias_tile ? D : tight_head_dim(D, p.d_qk, p.d_v);
    // ALiBi at 96: dK / dV of long tiles, one to a CU, by the pair of waves of 128, whose distances and slope gradient one wave
    // has to form beside everything else (us, at 96 -> at 128: M=N=2048 H=8 62 -> 59, with the gradient 69 -> 63, M=N=4096 H=4 129 ->
    // 114; at 1024 rows, H=32, 2 % the other way, at two tiles to a CU 26 %)
    if (kernel_dim == 96 && bias == 5 && (stages & 2) && p.M > 1024 && (int64_t)p.n_ntiles * p.B * p.H <= p.cus) {
        if (stages & 5) {
            const hipError_t e = launch_bwd_d<96>(p, dtype, bias, causal, dbias, stages & ~2, st);
            if (e != hipSuccess) return e;
        }
        return launch_bwd_d<128>(p, dtype, bias, causal, dbias, 2, st);
    }
    switch (kernel_dim) {
        case 16: return launch_bwd_d<16>(p, dtype, bias, causal, dbias, stages, st);
        case 32: return launch_bwd_d<32>(p, dtype, bias, causal, dbias, stages, st);
        case 64: return launch_bwd_d<64>(p, dtype, bias, causal, dbias, stages, st);
        case 96: return launch_bwd_d<96>(p, dtype, bias, causal, dbias, stages, st);
        case 128: return launch_bwd_d<128>(p, dtype, bias, causal, dbias, stages, st);
        case 256: return launch_bwd_d<256>(p, dtype, bias, causal, dbias, stages, st);
    }
    return hipErrorNotSupported;
}
static hipError_t launch_bwd_shared(const BwdParams& p, int D, int dtype, hipStream_t st) {
    switch (D) {
        case 16: return launch_bwd_shared_d<16>(p, dtype, st);
        case 32: return launch_bwd_shared_d<32>(p, dtype, st);
        case 64: return launch_bwd_shared_d<64>(p, dtype, st);
        case 128: return launch_bwd_shared_d<128>(p, dtype, st);
        case 256: return launch_bwd_shared_d<256>(p, dtype, st);
    }
    return hipErrorNotSupported;
}
// query rows per work-group of the forward and dQ kernels; keys per work-group of the dK/dV kernel
static int fwd_block_m() { return 128; }
static int bwd_block_n(int D) { return D > 128 ? 64 : 128; }  // keys per tile of the dK/dV kernel
}  // namespace fa

// Scratch of fa_bwd_noalloc: delta, one float per (batch, head, query row), in the first half; the
// partial sums of a reduced dbias in the second.  Every GPU the library
// runs on holds its own copy of this array until the process ends.  In host code the name is only
// a handle; the device address comes from hipGetSymbolAddress (scratch_on_current_device).
static __device__ __align__(256) float scratch[2 * FA_NOALLOC_MAX_ROWS];

namespace fa {

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static float* g_scratch_ptr[kMaxDevices];  // device address of `scratch`, per device

// Address of this device's copy of `scratch`, looked up once per device with that device current.
// This function has external linkage on purpose: the compiler gives a static device variable a
// symbol the runtime can find only when a host function with external linkage refers to it.
float* scratch_on_current_device() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
        g_scratch_ptr[dev] = static_cast<float*>(ptr);
    }
    return g_scratch_ptr[dev];
}

}  // namespace fa

namespace {

// Head dims of q / k and of v below the kernel's, p.D: whole 16-byte chunks.  (The kernels of head dim 256 form the
// offsets of their copies in the loop and take their full width only; the kernel of a shared bias's gradient has both
// operands of its products in LDS and so nothing to put against the missing columns.)
bool dims_ok(const fa_problem& p, int d_qk, int d_v) {
    if (d_qk == p.D && d_v == p.D) return true;
    return p.D <= 128 && d_qk >= 8 && d_v >= 8 && d_qk <= p.D && d_v <= p.D && d_qk % 8 == 0 && d_v % 8 == 0;
}

bool head_dim_ok(int d) { return d == 16 || d == 32 || d == 64 || d == 128 || d == 256; }

int check_problem(const fa_problem& p) {
    if (p.B < 1 || p.H < 1 || p.M < 1 || p.N < 1) return FA_ERR_SHAPE;
    if (!head_dim_ok(p.D)) return FA_ERR_HEAD_DIM;
    if (p.dtype != FA_F16 && p.dtype != FA_BF16) return FA_ERR_DTYPE;
    if (p.bias_dtype < FA_BIAS_NONE || p.bias_dtype > FA_BIAS_ALIBI) return FA_ERR_DTYPE;
    if (p.causal && p.M != p.N) return FA_ERR_SHAPE;
    // row indices times four (the LSE and delta vectors) are formed in 32 bits
    if (p.M >= (1 << 28) || p.N >= (1 << 28)) return FA_ERR_SHAPE;
    // a grid is one-dimensional: tiles * B * H must fit in 31 bits
    if ((int64_t)((p.M + 63) / 64 + (p.N + 63) / 64) * p.B * p.H >= (1ll << 31)) return FA_ERR_SHAPE;
    return FA_OK;
}

// 16-byte rule for a (B, seq, H, D) tensor of 2-byte elements; strides of extent-1 dims are free
// (FA_OK, FA_ERR_HEAD_STRIDE or FA_ERR_LAYOUT)
int qkv_layout(const void* ptr, const int64_t s[4], int nb, int ns, int nh) {
    if (s[3] != 1) return FA_ERR_HEAD_STRIDE;
    if (reinterpret_cast<uintptr_t>(ptr) % 16 != 0) return FA_ERR_LAYOUT;
    if (nb > 1 && s[0] % 8 != 0) return FA_ERR_LAYOUT;
    if (ns > 1 && s[1] % 8 != 0) return FA_ERR_LAYOUT;
    if (nh > 1 && s[2] % 8 != 0) return FA_ERR_LAYOUT;
    // the kernels form 32-bit byte offsets inside a tile of up to 128 rows
    if (ns > 1 && (s[1] < 0 || s[1] >= (1 << 23))) return FA_ERR_LAYOUT;
    return FA_OK;
}
// the first complaint among several tensors
int first_bad(std::initializer_list<int> sts) {
    for (int s : sts)
        if (s != FA_OK) return s;
    return FA_OK;
}

fa::Strides3 s3(const int64_t s[4]) { return fa::Strides3{s[0], s[1], s[2]}; }
fa::Strides4 s4(const int64_t s[4]) { return fa::Strides4{s[0], s[1], s[2], s[3]}; }

int bias_elem_size(int bias_dtype) {
    switch (bias_dtype) {
        case FA_BIAS_BOOL: return 1;
        case FA_BIAS_F16:
        case FA_BIAS_BF16: return 2;
        case FA_BIAS_F32: return 4;
    }
    return 0;
}

// rows of bias may be fetched with aligned 16-byte loads
bool bias_vec_ok(const void* ptr, const int64_t s[4], const fa_problem& p) {
    int es = bias_elem_size(p.bias_dtype);
    if (es == 0) return false;
    if (p.N > 1 && s[3] != 1) return false;
    if (reinterpret_cast<uintptr_t>(ptr) % 16 != 0) return false;
    if (p.B > 1 && (s[0] * es) % 16 != 0) return false;
    if (p.H > 1 && (s[1] * es) % 16 != 0) return false;
    if (p.M > 1 && (s[2] * es) % 16 != 0) return false;
    // A copy fetches whole 16-byte chunks: either the rows are whole chunks, or the row stride leaves
    // room for the last one (a padded row pitch, or a column slice of a wider tensor), so that the
    // bytes behind the last key of a row are readable; the kernels mask what they read there and write
    // a partial chunk of dbias element by element.
    const int64_t row_bytes = (int64_t)p.N * es, padded = (row_bytes + 15) & ~(int64_t)15;
    if (row_bytes != padded && !(p.M > 1 && s[2] * es >= padded)) return false;
    // one (batch, head) slice is addressed through a 32-bit buffer descriptor
    if (s[2] < 0 || (int64_t)(p.M - 1) * s[2] * es + padded >= (1ll << 31)) return false;
    return true;
}

// How the kernels fetch the rows of a bias: 1 in aligned 16-byte chunks; 2 (fp32, head dims up to 64) 4 bytes to a lane, whatever
// multiple of 4 bytes a row starts at; 0 element by element.
int bias_rows(const void* ptr, const int64_t s[4], const fa_problem& p) {
    if (bias_vec_ok(ptr, s, p)) return 1;
    if (p.bias_dtype != FA_BIAS_F32 || p.D > 64 || (p.N > 1 && s[3] != 1) || reinterpret_cast<uintptr_t>(ptr) % 4 != 0) return 0;
    // (offsets from the first row of a (batch, head) slice are formed in 32 bits)
    return s[2] >= 0 && ((int64_t)(p.M - 1) * s[2] + p.N) * 4 < (1ll << 31) ? 2 : 0;
}

// rows of bias or dbias may be accessed four elements at a time, at multiples of four
bool bias_quads_ok(const void* ptr, const int64_t s[4], const fa_problem& p) {
    const int es = bias_elem_size(p.bias_dtype);
    return es > 1 && s[3] == 1 && reinterpret_cast<uintptr_t>(ptr) % (4 * es) == 0 && (p.B == 1 || s[0] % 4 == 0) &&
           (p.H == 1 || s[1] % 4 == 0) && (p.M == 1 || s[2] % 4 == 0);
}

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// With FA_MI355_VERBOSE set in the environment, says once per process on stderr when a bias cannot
// take the 16-byte copy path and the kernels fall back to reading or writing it element by element
// (much slower; the rules are in the header).
void note_slow_bias(const char* what, const void* ptr, const int64_t s[4], const fa_problem& p) {
    static std::atomic<bool> said{false};
    if (!std::getenv("FA_MI355_VERBOSE") || said.exchange(true)) return;
    std::fprintf(stderr,
                 "libfa_mi355: %s takes the element-wise path (pointer %p, strides %lld/%lld/%lld/%lld elements, N = %d): "
                 "needs unit key stride, 16-byte aligned base and B/H/M strides, rows of whole 16-byte chunks (or a "
                 "row stride that covers the last chunk) and (batch, head) slices below 2 GiB\n",
                 what, ptr, (long long)s[0], (long long)s[1], (long long)s[2], (long long)s[3], p.N);
}

// the two parts of the backward scratch, in floats: delta, and the partial sums of a reduced
// dbias (column sums per (batch, head, key), or slope gradients per (batch, head, key tile, wave))
size_t delta_floats(const fa_problem& p) { return (size_t)p.B * p.H * p.M; }
size_t partial_floats(const fa_problem& p) {
    const size_t tiles4 = (size_t)((p.N + fa::bwd_block_n(p.D) - 1) / fa::bwd_block_n(p.D)) * (fa::bwd_block_n(p.D) / 32);
    return (size_t)p.B * p.H * ((size_t)p.N > tiles4 ? (size_t)p.N : tiles4);
}

// Compute units of the current device (looked up once per device; 256, an MI355X, when no device
// can be asked: the size queries must also work where no GPU is present).
int compute_units() {
    static std::atomic<int> cached[fa::kMaxDevices];
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= fa::kMaxDevices) return 256;
    int n = cached[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

// Keys of a query tile split between work-groups when the query tiles alone leave the GPU half empty
// (fewer than two work-groups per CU): as many splits as it takes to get there, each with at least 1024 keys, or
// 512 with a bias, whose steps cost more (D=64, byte mask, B=1 H=8 M=512 N=2048, shares of 512 / of 1024 keys: forward
// 19 / 25 us, dQ 19 / 27; bf16 tile 18 / 23 and 18 / 24; bf16 row 17 / 21 and 18 / 23; B=1 H=16 M=N=1024, a
// row: forward 19 / 17, dQ 20 / 20).  A few short tiles (at most one per four CUs, at most 256 query rows) go down
// to shares of 256 keys: their shares of the output are small next to the keys that they have read, and without
// that a token decoded against a long cache runs on a handful of CUs.  Beyond 32 shares the merge costs more than the
// last of them bring.  One query row, D = 128, us per call, at most 4 shares of at least 1024 / this rule / 64 shares
// allowed: B=1 H=8 N=1024 19.2 / 11.9 / 11.9, N=4096 22.8 / 15.4 / 15.4, N=16384 87 / 30 / 38.  Where the line lies: 256 keys
// at 256 tiles (B=16 H=16 N=700 D=64) 16.0 -> 18.5, at 1024 rows (B=2 H=8 M=N=1024 D=64) 14.8 -> 18.2.
// The answer depends on the current device (its CU
// count): a size query and the launch it sizes must run with the same device current.
struct FwdSplit {
    int n_splits, keys_per_split;
};
FwdSplit fwd_split(const fa_problem& p) {
    if (p.causal) return {1, 0};
    const int64_t wgs = (int64_t)((p.M + fa::fwd_block_m() - 1) / fa::fwd_block_m()) * p.B * p.H;
    const int64_t full = 2 * (int64_t)compute_units();
    if (wgs >= full) return {1, 0};
    const int unit = p.bias_dtype == FA_BIAS_NONE ? 64 : 32;  // keys are dealt in these
    const int n_units = (p.N + unit - 1) / unit;
    int s = (int)(full / wgs);
    s = s > 32 ? 32 : s;
    const int min_units = p.M <= 256 && 8 * wgs <= full ? 256 / unit : 16;
    while (s > 1 && n_units / s < min_units) s--;
    if (s <= 1) return {1, 0};
    const int keys = ((n_units + s - 1) / s * unit + 63) / 64 * 64;  // whole steps of every kernel tiling
    return {(p.N + keys - 1) / keys, keys};                        // (rounded up, they may need fewer shares: none is empty)
}

// the shares of dq of a dQ kernel that splits its keys like the forward (0 when it does not)
size_t dq_share_bytes(const fa_problem& p) {
    const FwdSplit s = fwd_split(p);
    return s.n_splits <= 1 ? 0 : align256((size_t)s.n_splits * p.B * p.H * p.M * p.D * sizeof(float));
}

// How dbias is laid out: 0 none, 1 dense (B, H, M, N), 2 summed over the query rows in the kernels, 3 of a bias that
// batches or heads share; -1 = not acceptable
int dbias_mode(const fa_bwd_args* a) {
    const fa_problem& p = a->p;
    if (!a->dbias) return 0;
    if (p.bias_dtype == FA_BIAS_ALIBI) return 2;
    const int64_t* s = a->dbias_strides;
    const bool red_b = p.B > 1 && s[0] == 0, red_h = p.H > 1 && s[1] == 0, red_m = p.M > 1 && s[2] == 0;
    if (p.N > 1 && s[3] == 0) return -1;  // nothing sums over the keys: they would all store to one address
    if (!red_b && !red_h && !red_m) return 1;
    if (!red_m && p.M > 1) {
        // the bias itself must be the one that is shared: its tile is read once for all pairs
        return (red_b && a->bias_strides[0] != 0) || (red_h && a->bias_strides[1] != 0) ? -1 : 3;
    }
    return 2;
}

// tiles of the gradient of a shared bias, over all of its slices
int64_t shared_tiles(const fa_bwd_args* a) {
    const fa_problem& p = a->p;
    return (int64_t)((p.M + fa::kSharedTileM - 1) / fa::kSharedTileM) * ((p.N + fa::kSharedTileN - 1) / fa::kSharedTileN) *
           (a->dbias_strides[0] == 0 ? 1 : p.B) * (a->dbias_strides[1] == 0 ? 1 : p.H);
}
// Work-groups that split the (batch, head) pairs of a tile of a shared bias's gradient between them: as many as fill
// the GPU, one per CU (LDS).
int shared_splits(const fa_bwd_args* a) {
    const fa_problem& p = a->p;
    const bool red_b = a->dbias_strides[0] == 0, red_h = a->dbias_strides[1] == 0;
    const int64_t tiles = shared_tiles(a);
    const int64_t pairs = (int64_t)(red_b ? p.B : 1) * (red_h ? p.H : 1);
    int64_t n = compute_units() / tiles;
    n = n < pairs ? n : pairs;
    return n < 1 ? 1 : (int)n;
}
// the shares of such a gradient in fp32, whole tiles (0 when nothing is split)
size_t shared_share_bytes(const fa_bwd_args* a) {
    if (dbias_mode(a) != 3) return 0;
    const int n = shared_splits(a);
    if (n == 1) return 0;
    return align256((size_t)shared_tiles(a) * n * fa::kSharedTileM * fa::kSharedTileN * sizeof(float));
}

}  // namespace

extern "C" {

int fa_abi_version(void) { return FA_ABI_VERSION; }

const char* fa_strerror(int status) {
    switch (status) {
        case FA_OK: return "ok";
        case FA_ERR_NULL: return "a required pointer is NULL";
        case FA_ERR_SHAPE: return "bad shape: a dimension is < 1, too large, or causal with M != N";
        case FA_ERR_HEAD_DIM: return "head dimension must be one of 16, 32, 64, 128, 256; d_qk and d_v that equal it, or (up to 128, not "
                                       "with the gradient of a bias that batches or heads share) multiples of 8 below it";
        case FA_ERR_DTYPE: return "unsupported dtype / bias dtype (or dbias requested for a bool bias)";
        case FA_ERR_LAYOUT:
            return "layout: head-dim stride must be 1 and pointers/strides 16-byte aligned; a dbias must not be broadcast over "
                   "the keys, and where it is broadcast over batches or heads but not over the query rows, the bias must be too";
        case FA_ERR_WORKSPACE: return "workspace is NULL, misaligned or smaller than fa_fwd_workspace_bytes() / fa_bwd_args_workspace_bytes()";
        case FA_ERR_UNSUPPORTED: return "combination not built into this library";
        case FA_ERR_LAUNCH: return "HIP kernel launch failed";
        case FA_ERR_TOO_LARGE: return "fa_bwd_noalloc: the problem exceeds FA_NOALLOC_MAX_ROWS";
        case FA_ERR_HEAD_STRIDE:
            return "the head-dim stride of q, k, v, o, do, dq, dk and dv must be 1: make the tensor contiguous first";
    }
    return "unknown status";
}

size_t fa_fwd_workspace_bytes(const fa_problem* p) {
    if (!p || check_problem(*p) != FA_OK) return 0;
    const FwdSplit s = fwd_split(*p);
    if (s.n_splits <= 1) return 0;
    const size_t rows = (size_t)p->B * p->H * p->M;
    return align256((size_t)s.n_splits * rows * p->D * sizeof(float)) + align256((size_t)s.n_splits * rows * sizeof(float));
}

int fa_fwd(const fa_fwd_args* a, void* stream) { return a ? fa_fwd_dims(a, a->p.D, a->p.D, stream) : FA_ERR_NULL; }

int fa_fwd_dims(const fa_fwd_args* a, int d_qk, int d_v, void* stream) {
    if (!a) return FA_ERR_NULL;
    const fa_problem& p = a->p;
    int st = check_problem(p);
    if (st != FA_OK) return st;
    if (!dims_ok(p, d_qk, d_v)) return FA_ERR_HEAD_DIM;
    if (!a->q || !a->k || !a->v || !a->o || !a->lse) return FA_ERR_NULL;
    if ((p.bias_dtype != FA_BIAS_NONE) != (a->bias != nullptr)) return FA_ERR_NULL;
    st = first_bad({qkv_layout(a->q, a->q_strides, p.B, p.M, p.H), qkv_layout(a->k, a->k_strides, p.B, p.N, p.H),
                    qkv_layout(a->v, a->v_strides, p.B, p.N, p.H), qkv_layout(a->o, a->o_strides, p.B, p.M, p.H)});
    if (st != FA_OK) return st;

    fa::FwdParams k{};
    k.q = a->q; k.k = a->k; k.v = a->v; k.bias = a->bias; k.o = a->o; k.lse = a->lse;
    k.sq = s3(a->q_strides); k.sk = s3(a->k_strides); k.sv = s3(a->v_strides); k.so = s3(a->o_strides);
    k.B = p.B; k.H = p.H; k.M = p.M; k.N = p.N;
    k.sm_scale = p.sm_scale;
    k.d_qk = d_qk; k.d_v = d_v; k.qk_inv = (256 + d_qk / 8 - 1) / (d_qk / 8);
    if (a->bias && p.bias_dtype != FA_BIAS_ALIBI) {
        k.sbias = s4(a->bias_strides);
        k.bias_vec = bias_rows(a->bias, a->bias_strides, p);
        if (!k.bias_vec) note_slow_bias("bias", a->bias, a->bias_strides, p);
    }
    k.n_mtiles = (p.M + fa::fwd_block_m() - 1) / fa::fwd_block_m();
    k.n_splits = 1;
    if (a->workspace) {
        const size_t need = fa_fwd_workspace_bytes(&p);
        if (need > 0) {
            if (a->workspace_bytes < need || reinterpret_cast<uintptr_t>(a->workspace) % 256 != 0) return FA_ERR_WORKSPACE;
            const FwdSplit s = fwd_split(p);
            const size_t rows = (size_t)p.B * p.H * p.M;
            k.n_splits = s.n_splits;
            k.keys_per_split = s.keys_per_split;
            k.part_o = a->workspace;
            k.part_lse = reinterpret_cast<float*>(static_cast<char*>(a->workspace) + align256((size_t)s.n_splits * rows * p.D * sizeof(float)));
        }
    }
    // a bias that does not depend on the query row and whose keys fit the kernel's LDS row
    if (a->bias && p.bias_dtype >= FA_BIAS_BOOL && p.bias_dtype <= FA_BIAS_F32 && (p.M == 1 || a->bias_strides[2] == 0) &&
        (k.n_splits > 1 ? k.keys_per_split : p.N) <= fa::kRowBiasKeys)
        k.row_bias_kind = p.bias_dtype;
    hipError_t e = fa::launch_fwd(k, p.D, p.dtype, p.bias_dtype, p.causal != 0, static_cast<hipStream_t>(stream));
    if (e == hipErrorNotSupported) return FA_ERR_UNSUPPORTED;
    return e == hipSuccess ? FA_OK : FA_ERR_LAUNCH;
}

size_t fa_bwd_workspace_bytes(const fa_problem* p) {
    if (!p || check_problem(*p) != FA_OK) return 0;
    return align256(delta_floats(*p) * sizeof(float)) + align256(partial_floats(*p) * sizeof(float)) + dq_share_bytes(*p);
}

size_t fa_bwd_args_workspace_bytes(const fa_bwd_args* a) {
    if (!a) return 0;
    const size_t base = fa_bwd_workspace_bytes(&a->p);
    return base == 0 ? 0 : base + shared_share_bytes(a);
}

}  // extern "C"

namespace {

// `delta` NULL: the scratch is the caller's workspace; else the workspace fields are ignored
int bwd_enqueue(const fa_bwd_args* a, int d_qk, int d_v, void* stream, int stages, float* delta) {
    if (!a) return FA_ERR_NULL;
    if (stages <= 0 || (stages & ~(FA_STAGE_ALL | FA_STAGE_DQ_FROM_DBIAS))) return FA_ERR_UNSUPPORTED;
    if ((stages & FA_STAGE_DQ_FROM_DBIAS) && !(stages & FA_STAGE_DQ)) return FA_ERR_UNSUPPORTED;
    const fa_problem& p = a->p;
    int st = check_problem(p);
    if (st != FA_OK) return st;
    if (!dims_ok(p, d_qk, d_v)) return FA_ERR_HEAD_DIM;
    if (!a->q || !a->k || !a->v || !a->o || !a->dout || !a->lse) return FA_ERR_NULL;
    // outputs of stages that do not run may be NULL
    const bool need_dq = (stages & FA_STAGE_DQ) != 0, need_dkv = (stages & FA_STAGE_MAIN) != 0;
    if ((need_dq && !a->dq) || (need_dkv && (!a->dk || !a->dv))) return FA_ERR_NULL;
    if ((p.bias_dtype != FA_BIAS_NONE) != (a->bias != nullptr)) return FA_ERR_NULL;
    if (a->dbias && (p.bias_dtype == FA_BIAS_NONE || p.bias_dtype == FA_BIAS_BOOL)) return FA_ERR_DTYPE;
    const int db_mode = dbias_mode(a);
    if (db_mode < 0) return FA_ERR_LAYOUT;
    if (db_mode == 3 && (d_qk != p.D || d_v != p.D)) return FA_ERR_HEAD_DIM;
    if (db_mode == 3 && shared_tiles(a) >= (1ll << 26)) return FA_ERR_SHAPE;  // its grid is one-dimensional too
    st = first_bad({qkv_layout(a->q, a->q_strides, p.B, p.M, p.H), qkv_layout(a->k, a->k_strides, p.B, p.N, p.H),
                    qkv_layout(a->v, a->v_strides, p.B, p.N, p.H), qkv_layout(a->o, a->o_strides, p.B, p.M, p.H),
                    qkv_layout(a->dout, a->do_strides, p.B, p.M, p.H),
                    need_dq ? qkv_layout(a->dq, a->dq_strides, p.B, p.M, p.H) : FA_OK,
                    need_dkv ? qkv_layout(a->dk, a->dk_strides, p.B, p.N, p.H) : FA_OK,
                    need_dkv ? qkv_layout(a->dv, a->dv_strides, p.B, p.N, p.H) : FA_OK});
    if (st != FA_OK) return st;
    float* partials = nullptr;
    int dq_splits = 1, dq_keys = 0;  // (the entry point without allocations does not split: its scratch is small)
    void* part_dq = nullptr;
    int splits = 1;  // work-groups per tile of a shared bias's gradient
    if (!delta) {
        const size_t share_bytes = need_dkv ? shared_share_bytes(a) : 0;
        size_t need = fa_bwd_workspace_bytes(&p) + share_bytes;
        if (!a->workspace || a->workspace_bytes < need || reinterpret_cast<uintptr_t>(a->workspace) % 256 != 0)
            return FA_ERR_WORKSPACE;
        delta = static_cast<float*>(a->workspace);
        partials = reinterpret_cast<float*>(static_cast<char*>(a->workspace) + align256(delta_floats(p) * sizeof(float)));
        if (dq_share_bytes(p) > 0) {
            const FwdSplit s = fwd_split(p);
            dq_splits = s.n_splits;
            dq_keys = s.keys_per_split;
            part_dq = reinterpret_cast<char*>(partials) + align256(partial_floats(p) * sizeof(float));
        }
        if (share_bytes > 0) {
            splits = shared_splits(a);
            // (a shared bias has no column sums: its shares stand behind everything else)
            partials = reinterpret_cast<float*>(static_cast<char*>(a->workspace) + fa_bwd_workspace_bytes(&p));
        }
    } else {
        partials = delta + FA_NOALLOC_MAX_ROWS;
    }

    fa::BwdParams k{};
    k.q = a->q; k.k = a->k; k.v = a->v; k.o = a->o; k.dout = a->dout; k.bias = a->bias; k.lse = a->lse;
    k.dq = a->dq; k.dk = a->dk; k.dv = a->dv; k.dbias = a->dbias;
    k.delta = delta;
    k.partials = partials;
    k.dq_splits = dq_splits; k.dq_keys_per_split = dq_keys; k.part_dq = part_dq;
    k.sq = s3(a->q_strides); k.sk = s3(a->k_strides); k.sv = s3(a->v_strides); k.so = s3(a->o_strides);
    k.sdo = s3(a->do_strides); k.sdq = s3(a->dq_strides); k.sdk = s3(a->dk_strides); k.sdv = s3(a->dv_strides);
    if (a->bias && p.bias_dtype != FA_BIAS_ALIBI) {
        k.sbias = s4(a->bias_strides);
        k.bias_vec = bias_rows(a->bias, a->bias_strides, p);
    }
    // a bias that does not depend on the query row: the dK/dV kernel keeps it in one register per key
    if (a->bias && p.bias_dtype >= FA_BIAS_BOOL && p.bias_dtype <= FA_BIAS_F32 && (p.M == 1 || a->bias_strides[2] == 0))
        k.row_bias_kind = p.bias_dtype;
    if (a->dbias && p.bias_dtype != FA_BIAS_ALIBI) {
        k.sdbias = s4(a->dbias_strides);
        k.dbias_vec = db_mode == 1 && bias_vec_ok(a->dbias, a->dbias_strides, p) ? 1 : 0;
        if (db_mode == 1 && !k.dbias_vec) note_slow_bias("dbias", a->dbias, a->dbias_strides, p);
    }
    k.B = p.B; k.H = p.H; k.M = p.M; k.N = p.N;
    k.sm_scale = p.sm_scale;
    k.d_qk = d_qk; k.d_v = d_v; k.qk_inv = (256 + d_qk / 8 - 1) / (d_qk / 8);
    int bn = fa::bwd_block_n(p.D);
    if (bn <= 0) return FA_ERR_UNSUPPORTED;
    k.n_ntiles = (p.N + bn - 1) / bn;
    k.waves_per_role = bn / 32;
    k.n_mtiles = (p.M + fa::fwd_block_m() - 1) / fa::fwd_block_m();
    k.causal = p.causal != 0; k.bias_kind = p.bias_dtype; k.shared_splits = splits; k.cus = compute_units();
    if (db_mode == 3) {
        k.shared_tiles = (int)shared_tiles(a);
        k.bias_quads = bias_quads_ok(a->bias, a->bias_strides, p) ? 1 : 0;
        k.dbias_quads = bias_quads_ok(a->dbias, a->dbias_strides, p) ? 1 : 0;
    }
    hipError_t e = fa::launch_bwd(k, p.D, p.dtype, p.bias_dtype, p.causal != 0, db_mode, stages,
                                  static_cast<hipStream_t>(stream));
    if (e == hipSuccess && db_mode == 3 && need_dkv) e = fa::launch_bwd_shared(k, p.D, p.dtype, static_cast<hipStream_t>(stream));
    if (e == hipErrorNotSupported) return FA_ERR_UNSUPPORTED;
    return e == hipSuccess ? FA_OK : FA_ERR_LAUNCH;
}

}  // namespace

extern "C" {

int fa_bwd_stages_dims(const fa_bwd_args* a, int d_qk, int d_v, void* stream, int stages) {
    return bwd_enqueue(a, d_qk, d_v, stream, stages, nullptr);
}

int fa_bwd_stages(const fa_bwd_args* a, void* stream, int stages) {
    return a ? bwd_enqueue(a, a->p.D, a->p.D, stream, stages, nullptr) : FA_ERR_NULL;
}

int fa_bwd(const fa_bwd_args* a, void* stream) { return fa_bwd_stages(a, stream, FA_STAGE_ALL); }

int fa_bwd_noalloc(const fa_bwd_args* a, void* stream) {
    if (!a) return FA_ERR_NULL;
    int st = check_problem(a->p);
    if (st != FA_OK) return st;
    if (delta_floats(a->p) > (size_t)FA_NOALLOC_MAX_ROWS || partial_floats(a->p) > (size_t)FA_NOALLOC_MAX_ROWS)
        return FA_ERR_TOO_LARGE;
    float* delta = fa::scratch_on_current_device();
    if (!delta) return FA_ERR_LAUNCH;
    return bwd_enqueue(a, a->p.D, a->p.D, stream, FA_STAGE_ALL, delta);
}

}  // extern "C"
