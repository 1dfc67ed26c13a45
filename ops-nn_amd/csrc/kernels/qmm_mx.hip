// MX quantized matmul: fp4 e2m1 (or fp8 e4m3) operands with one e8m0 scale per 32 K elements.
//
//   out[m,n] = cast( sum_k (x1[m,k] * 2^(s1[m,k/32]-127)) * (x2[k,n] * 2^(s2[k/32,n]-127)) + bias[n] )
//
// Formula and scale layouts: matmul/quant_batch_matmul_v3/tests/assets/qbmmv3_kernel_golden.py:153-234; the
// device counterpart in the reference is the MX block-mmad (matmul/common/cmct/block/block_mmad_mx.h).
// Here the contraction and the scaling are one instruction, v_mfma_scale_f32_32x32x64_f8f6f4: each lane hands
// the matrix core its 32 K elements together with the e8m0 byte that scales exactly those 32 elements, so the
// MX block size (32) and the hardware operand block coincide and no dequantised copy is ever formed.
//
// Few rows of fp4: the stream kernel of qmm_mxfp4_rows.hip, whatever K's tail.
// Fast paths: operands and scales K-contiguous, 16-bit or fp32 output.  fp4: qgemm_core.hip.h, MODE_MXFP4 (256 x 256 tiles: K tiles of
// 256 elements, a K that is no whole pair of them ending in zeros inside the kernel; 128 x 128 tiles: of 128); fp8: the MX mode of the
// kernel in qmm_fp8_block.hip.  An N-contiguous x2 (data [K, N], scales [K/64, N, 2]) is first re-laid out into the workspace.
// K % 128 != 0 (K a whole number of 32-element blocks): both operands and both scale tables (x2's after that re-layout, if it was needed)
// are first copied into the workspace with K rounded up to 128, the new elements zero and their scales a repeat of the row's last one
// (zero products change no sum); the 256 x 256 fp4 tiles need the scale tables alone.  All of this is planned before the first
// pre-step is launched.  Everything else runs the plain kernel.
#include "launch.h"
#include "qgemm_core.hip.h"

namespace opsnn {

// dst[c, r] = src[r, c] for 16-bit elements: the paired e8m0 scales [K/64, N, 2] -> [N, K/64, 2].
__global__ __launch_bounds__(256) void transpose16_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst,
                                                          int64_t rows, int64_t cols)
{
    __shared__ uint16_t tile[32][33];
    const int64_t bz = blockIdx.z;
    src += bz * rows * cols;
    dst += bz * rows * cols;
    const int64_t r0 = (int64_t)blockIdx.y * 32, c0 = (int64_t)blockIdx.x * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int i = ty; i < 32; i += 8) {
        int64_t r = r0 + i, c = c0 + tx;
        tile[i][tx] = (r < rows && c < cols) ? src[r * cols + c] : 0;
    }
    __syncthreads();
    for (int i = ty; i < 32; i += 8) {
        int64_t c = c0 + i, r = r0 + tx;
        if (c < cols && r < rows) dst[c * rows + r] = tile[tx][i];
    }
}

}  // namespace opsnn
extern "C" int opsnnTranspose16(const void* src, void* dst, int64_t rows, int64_t cols, int64_t batch, void* stream)
{
    if (!src || !dst || rows <= 0 || cols <= 0 || batch <= 0 || batch > 65535) return -1;
    dim3 grid((unsigned)((cols + 31) / 32), (unsigned)((rows + 31) / 32), (unsigned)batch);
    if (grid.y > 65535u) return -2;
    hipLaunchKernelGGL(opsnn::transpose16_kernel, grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t*)src, (uint16_t*)dst, rows, cols);
    return (int)hipGetLastError();
}
namespace opsnn {

static inline uint64_t align_up(uint64_t v, uint64_t a) { return (v + a - 1) / a * a; }
extern "C" bool opsnn_force_plain();   // dispatch.hip

// ---- K % 128 != 0 (whole MX blocks: K % 32 == 0) ----
// rows of kb bytes (pitch ld) -> rows of kbp bytes, the tail filled with the byte `fill`; E = bytes per thread.  E == 16:
// kb is a multiple of 16.  E == 2 (scale rows): kb counts the bytes that scale existing elements; the second byte of a
// source pair may lie past it (K % 64 == 32) and is replaced like the rest of the tail, whatever the caller left there.
// Scale tails repeat the row's last valid byte; data tails are zero.
template <int E>
__global__ __launch_bounds__(256) void mx_pad_rows_kernel(const uint8_t* __restrict__ src, int64_t ld, int64_t bs, uint8_t* __restrict__ dst,
                                                          int64_t rows, int64_t kb, int64_t kbp, uint32_t fill)
{
    const int64_t c = (int64_t)blockIdx.x * 64 + (threadIdx.x & 63), r = (int64_t)blockIdx.y * 4 + (threadIdx.x >> 6);
    if (c * E >= kbp || r >= rows) return;
    const uint8_t* s = src + (int64_t)blockIdx.z * bs + r * ld + c * E;
    uint8_t* d = dst + ((int64_t)blockIdx.z * rows + r) * kbp + c * E;
    if constexpr (E == 16) {
        *(uint4*)d = c * E < kb ? *(const uint4*)s : make_uint4(fill, fill, fill, fill);
    } else {
        // the tail repeats the row's last valid scale byte (its elements are zero, so any finite scale will do; a row whose
        // scales are finite gets no other kind)
        (void)fill;
        const uint32_t last = (src + (int64_t)blockIdx.z * bs + r * ld)[kb - 1];
        uint16_t v = (uint16_t)(last | (last << 8));
        if (c * 2 + 1 < kb) v = *(const uint16_t*)s;
        else if (c * 2 < kb) v = (uint16_t)((v & 0xFF00u) | s[0]);
        *(uint16_t*)d = v;
    }
}

struct MxPad {
    int64_t Kp, nb1, nb2, snb1, snb2;
    uint64_t o_x2, o_s1, o_s2, total;
};

// Whether the padding pre-step serves this call, and its workspace layout.
static bool mx_pad_layout(const OpsnnQmmArgs& a, MxPad& L)
{
    const bool fp4 = a.x1_dtype == DT_E2M1 && a.x2_dtype == DT_E2M1, fp8 = a.x1_dtype == DT_E4M3 && a.x2_dtype == DT_E4M3;
    const bool a8w4 = a.x1_dtype == DT_E4M3 && a.x2_dtype == DT_E2M1;   // the matrix-core kernel of that mode: 16-bit output, fp32 or 16-bit bias
    if ((!fp4 && !fp8 && !a8w4) || a.K % 128 == 0 || a.K % 32 != 0 || a.M * a.N < 64 * 64) return false;
    if (a.out_dtype != DT_BF16 && a.out_dtype != DT_F16 && !(a.out_dtype == DT_F32 && !a8w4)) return false;
    if (a.bias && a.bias_dtype != DT_F32 && !(a8w4 && (a.bias_dtype == DT_BF16 || a.bias_dtype == DT_F16))) return false;
    const int64_t epb1 = a.x1_dtype == DT_E2M1 ? 2 : 1, epb2 = a.x2_dtype == DT_E2M1 ? 2 : 1, ks = (a.K + 63) / 64;   // elements per byte; scale pairs per row
    if (a.x1.col_stride != 1 || a.x2.row_stride != 1) return false;
    if (a.x1_scale_mat.col_stride != 2 || a.x1_scale_mat.row_stride != ks * 2) return false;
    if (a.x2_scale_mat.col_stride != 2 || a.x2_scale_mat.row_stride != ks * 2) return false;
    if (a.x1.batch_stride < 0 || a.x2.batch_stride < 0 || a.x1_scale_mat.batch_stride < 0 || a.x2_scale_mat.batch_stride < 0) return false;
    // 16-byte pieces of the data rows, 2-byte pieces of the scale rows
    if (((uintptr_t)a.x1.ptr | (uintptr_t)a.x2.ptr | (uint64_t)(a.x1.row_stride / epb1) | (uint64_t)(a.x2.col_stride / epb2) |
         (uint64_t)(a.x1.batch_stride / epb1) | (uint64_t)(a.x2.batch_stride / epb2)) % 16) return false;
    if (((uintptr_t)a.x1_scale_mat.ptr | (uintptr_t)a.x2_scale_mat.ptr | (uint64_t)a.x1_scale_mat.batch_stride | (uint64_t)a.x2_scale_mat.batch_stride) % 2) return false;
    if ((a.M + 3) / 4 > 65535 || (a.N + 3) / 4 > 65535) return false;
    L.Kp = (a.K + 127) / 128 * 128;
    L.nb1 = a.x1.batch_stride == 0 && a.batch > 1 ? 1 : a.batch;
    L.nb2 = a.x2.batch_stride == 0 ? 1 : a.batch;
    L.snb1 = a.x1_scale_mat.batch_stride == 0 && a.batch > 1 ? 1 : a.batch;
    L.snb2 = a.x2_scale_mat.batch_stride == 0 ? 1 : a.batch;
    const uint64_t ksp = (uint64_t)L.Kp / 64;
    L.o_x2 = align_up((uint64_t)L.nb1 * a.M * (L.Kp / epb1), 256);
    L.o_s1 = L.o_x2 + align_up((uint64_t)L.nb2 * a.N * (L.Kp / epb2), 256);
    L.o_s2 = L.o_s1 + align_up((uint64_t)L.snb1 * a.M * ksp * 2, 256);
    L.total = L.o_s2 + align_up((uint64_t)L.snb2 * a.N * ksp * 2, 256);
    return true;
}

// The scale tables alone, both in one launch (rows of x1's, then of x2's along grid.x, which takes their sum): for fp4 on the tiles that end a K inside a
// tile by themselves, whose scales come in whole words.
__global__ __launch_bounds__(256) void mx_pad_scales_kernel(const uint8_t* __restrict__ s1, int64_t bs1, uint8_t* __restrict__ d1, int64_t rows1, int64_t nb1,
                                                            const uint8_t* __restrict__ s2, int64_t bs2, uint8_t* __restrict__ d2, int64_t rows2, int64_t nb2,
                                                            int64_t ld, int64_t kb, int64_t kbp)
{
    const int64_t c = (int64_t)blockIdx.y * 64 + (threadIdx.x & 63), b = blockIdx.z;
    int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const bool second = r >= rows1;
    if (second) r -= rows1;
    if (c * 2 >= kbp || r >= (second ? rows2 : rows1) || b >= (second ? nb2 : nb1)) return;
    const uint8_t* s = (second ? s2 + b * bs2 : s1 + b * bs1) + r * ld;
    uint8_t* d = (second ? d2 + b * rows2 * kbp : d1 + b * rows1 * kbp) + r * kbp + 2 * c;
    const uint8_t last = s[kb - 1];
    d[0] = 2 * c < kb ? s[2 * c] : last;
    d[1] = 2 * c + 1 < kb ? s[2 * c + 1] : last;
}
static int mx_pad_scales(OpsnnQmmArgs& a, const MxPad& L, hipStream_t st)
{
    if (!a.workspace || (uintptr_t)a.workspace % 16) return OPSNN_NOT_TAKEN;
    uint8_t* w = (uint8_t*)a.workspace;
    const int64_t ksp2 = L.Kp / 64 * 2, nb = L.snb1 > L.snb2 ? L.snb1 : L.snb2;
    const dim3 grid((unsigned)((a.M + a.N + 3) / 4), (unsigned)((ksp2 / 2 + 63) / 64), (unsigned)nb);
    hipLaunchKernelGGL(mx_pad_scales_kernel, grid, dim3(256), 0, st, (const uint8_t*)a.x1_scale_mat.ptr, a.x1_scale_mat.batch_stride, w + L.o_s1, a.M, L.snb1,
                       (const uint8_t*)a.x2_scale_mat.ptr, a.x2_scale_mat.batch_stride, w + L.o_s2, a.N, L.snb2, (a.K + 63) / 64 * 2, a.K / 32, ksp2);
    a.x1_scale_mat = OpsnnMat{w + L.o_s1, ksp2, 2, L.snb1 == 1 && a.batch > 1 ? 0 : a.M * ksp2};
    a.x2_scale_mat = OpsnnMat{w + L.o_s2, ksp2, 2, L.snb2 == 1 && a.batch > 1 ? 0 : a.N * ksp2};
    a.workspace = nullptr;
    return (int)hipGetLastError();
}

// Launches the four copies and rewrites `a` as the same call on the padded operands.
static int mx_pad_prestep(OpsnnQmmArgs& a, const MxPad& L, hipStream_t st)
{
    if (!a.workspace || (uintptr_t)a.workspace % 16) return OPSNN_NOT_TAKEN;
    const int64_t epb1 = a.x1_dtype == DT_E2M1 ? 2 : 1, epb2 = a.x2_dtype == DT_E2M1 ? 2 : 1;
    const int64_t kb1 = a.K / epb1, kbp1 = L.Kp / epb1, kb2 = a.K / epb2, kbp2 = L.Kp / epb2, ks2 = (a.K + 63) / 64 * 2, ksp2 = L.Kp / 64 * 2;
    const int64_t sv = a.K / 32;   // scale bytes per row that scale existing elements
    uint8_t* w = (uint8_t*)a.workspace;
    auto grid = [](int64_t pieces, int64_t rows, int64_t nb) { return dim3((unsigned)((pieces + 63) / 64), (unsigned)((rows + 3) / 4), (unsigned)nb); };
    hipLaunchKernelGGL(mx_pad_rows_kernel<16>, grid(kbp1 / 16, a.M, L.nb1), dim3(256), 0, st, (const uint8_t*)a.x1.ptr, a.x1.row_stride / epb1,
                       a.x1.batch_stride / epb1, w, a.M, kb1, kbp1, 0u);
    hipLaunchKernelGGL(mx_pad_rows_kernel<16>, grid(kbp2 / 16, a.N, L.nb2), dim3(256), 0, st, (const uint8_t*)a.x2.ptr, a.x2.col_stride / epb2,
                       a.x2.batch_stride / epb2, w + L.o_x2, a.N, kb2, kbp2, 0u);
    hipLaunchKernelGGL(mx_pad_rows_kernel<2>, grid(ksp2 / 2, a.M, L.snb1), dim3(256), 0, st, (const uint8_t*)a.x1_scale_mat.ptr, ks2,
                       a.x1_scale_mat.batch_stride, w + L.o_s1, a.M, sv, ksp2, 0x7f7fu);
    hipLaunchKernelGGL(mx_pad_rows_kernel<2>, grid(ksp2 / 2, a.N, L.snb2), dim3(256), 0, st, (const uint8_t*)a.x2_scale_mat.ptr, ks2,
                       a.x2_scale_mat.batch_stride, w + L.o_s2, a.N, sv, ksp2, 0x7f7fu);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    a.x1 = OpsnnMat{w, L.Kp, 1, L.nb1 == 1 && a.batch > 1 ? 0 : a.M * L.Kp};
    a.x2 = OpsnnMat{w + L.o_x2, 1, L.Kp, L.nb2 == 1 && a.batch > 1 ? 0 : a.N * L.Kp};
    a.x1_scale_mat = OpsnnMat{w + L.o_s1, ksp2, 2, L.snb1 == 1 && a.batch > 1 ? 0 : a.M * ksp2};
    a.x2_scale_mat = OpsnnMat{w + L.o_s2, ksp2, 2, L.snb2 == 1 && a.batch > 1 ? 0 : a.N * ksp2};
    a.K = L.Kp;
    a.workspace = nullptr;
    return 0;
}

uint64_t mx_exact_bytes(const OpsnnQmmArgs& a);           // qmm_fp8_exact.hip
int launch_mx_exact(const OpsnnQmmArgs& a, hipStream_t st, SplitK sk);

// ---- x2 stored [K, N] with N contiguous (data dense, scales [K/64, N, 2]) ----
// The kernels stream K-contiguous operands: data and scales are first re-laid out, per batch, at 256-byte aligned pitches.
struct MxRelayout {
    int64_t nb, snb;                 // batches of the data / of the scales (1 when every batch shares them)
    uint64_t data_one, scale_one, bytes;
};

static bool mx_relayout_layout(const OpsnnQmmArgs& a, MxRelayout& R)
{
    if (a.x2.row_stride == 1 || a.K == 1 || a.K % 32 != 0) return false;
    const int64_t ks = (a.K + 63) / 64, epb = a.x2_dtype == DT_E2M1 ? 2 : 1;
    if (a.x2.col_stride != 1 || a.x2.row_stride != a.N) return false;
    if (epb == 2 && (a.N & 1)) return false;   // the 4-bit transposition works on byte pairs
    if (a.x2_scale_mat.row_stride != 2 || a.x2_scale_mat.col_stride != a.N * 2) return false;
    if (a.x2.batch_stride != 0 && a.x2.batch_stride != a.K * a.N) return false;
    R.nb = a.x2.batch_stride == 0 ? 1 : a.batch;
    R.snb = a.x2_scale_mat.batch_stride == 0 ? 1 : a.batch;
    if (R.snb != 1 && a.x2_scale_mat.batch_stride != ks * a.N * 2) return false;
    if (R.nb > 65535 || R.snb > 65535) return false;
    R.data_one = align_up((uint64_t)a.N * a.K / epb, 256);
    R.scale_one = align_up((uint64_t)a.N * ks * 2, 256);
    R.bytes = R.data_one * (uint64_t)R.nb + R.scale_one * (uint64_t)R.snb;
    return true;
}

// `a` as the same call on the copies at `w` (which the passes of mx_relayout_run fill)
static void mx_relayout_view(OpsnnQmmArgs& a, const MxRelayout& R, char* w)
{
    const int64_t ks = (a.K + 63) / 64, epb = a.x2_dtype == DT_E2M1 ? 2 : 1;
    char* wscale = w + R.data_one * R.nb;
    a.x2.ptr = w; a.x2.row_stride = 1; a.x2.col_stride = a.K; a.x2.batch_stride = R.nb == 1 ? 0 : (int64_t)(R.data_one * epb);
    a.x2_scale_mat.ptr = wscale; a.x2_scale_mat.row_stride = ks * 2; a.x2_scale_mat.col_stride = 2;
    a.x2_scale_mat.batch_stride = R.snb == 1 ? 0 : (int64_t)R.scale_one;
}

static int mx_relayout_run(const OpsnnQmmArgs& a, const MxRelayout& R, char* w, hipStream_t st)
{
    const int64_t ks = (a.K + 63) / 64, epb = a.x2_dtype == DT_E2M1 ? 2 : 1;
    char* wscale = w + R.data_one * R.nb;
    for (int64_t b = 0; b < R.nb; b++) {  // per batch because of the aligned pitch
        const char* src = (const char*)a.x2.ptr + b * (a.K * a.N / epb);
        const int rc = epb == 2 ? opsnnTranspose4(src, w + b * R.data_one, a.K, a.N, 1, st) : opsnnTranspose8(src, w + b * R.data_one, a.K, a.N, 1, st);
        if (rc != 0) return rc;
    }
    for (int64_t b = 0; b < R.snb; b++) {
        dim3 grid((unsigned)((a.N + 31) / 32), (unsigned)((ks + 31) / 32), 1);
        hipLaunchKernelGGL(transpose16_kernel, grid, dim3(256), 0, st, (const uint16_t*)((const char*)a.x2_scale_mat.ptr + b * (ks * a.N * 2)),
                           (uint16_t*)(wscale + b * R.scale_one), ks, a.N);
    }
    return (int)hipGetLastError();
}

// ---- MXFP8 with fewer than 64 x 64 outputs and a last half K tile ----
// fp32 operands, x1 * 2^(a - 127) and x2 * 2^(b - 127) rounded nowhere down to scale byte 0, and fp32 sums, as on the plain kernel, which
// took these calls before (3 x 15168 x 1088 12.4 ms on one thread per output); in bf16, as the matrix instructions would have them,
// scale bytes 0 to 2 lose bits.  A workgroup per column of x2: its threads take pieces of 16 k in turns, multiply them with every row of x1,
// and their sums meet in LDS.  Bound by vector instructions, some 40 a piece and row, against x2's bytes at few rows.
template <int ROWS>
__global__ __launch_bounds__(256) void mxfp8_few_outputs_kernel(OpsnnQmmArgs a)
{
    __shared__ float red[4][ROWS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t n = blockIdx.x;
    const uint8_t* w = (const uint8_t*)a.x2.ptr + n * a.x2.col_stride;
    const uint8_t* ws = (const uint8_t*)a.x2_scale_mat.ptr + n * a.x2_scale_mat.row_stride;
    float acc[ROWS];
#pragma unroll
    for (int m = 0; m < ROWS; m++) acc[m] = 0.0f;
    auto widen = [](const uint4& v, float s, float (&o)[16]) {
        const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)d[i], false), hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)d[i], true);
            o[4 * i] = lo[0] * s; o[4 * i + 1] = lo[1] * s; o[4 * i + 2] = hi[0] * s; o[4 * i + 3] = hi[1] * s;
        }
    };
    const uint8_t* const x = (const uint8_t*)a.x1.ptr;
    const uint8_t* const xs = (const uint8_t*)a.x1_scale_mat.ptr;
    struct Pieces { uint4 w, x[ROWS]; uint8_t ws, xs[ROWS]; };
    auto fetch = [&](Pieces& f, int p) {
        f.w = *(const uint4*)(w + 16 * p);
        f.ws = ws[p >> 1];
#pragma unroll
        for (int m = 0; m < ROWS; m++) {
            const int64_t r = m < a.M ? m : a.M - 1;   // (past the last row: that row again, not stored)
            f.x[m] = *(const uint4*)(x + r * a.x1.row_stride + 16 * p);
            f.xs[m] = xs[r * a.x1_scale_mat.row_stride + (p >> 1)];
        }
    };
    auto multiply = [&](const Pieces& f) {
        float wf[16];
        widen(f.w, e8m0_to_f32(f.ws), wf);
#pragma unroll
        for (int m = 0; m < ROWS; m++) {
            float xf[16];
            widen(f.x[m], e8m0_to_f32(f.xs[m]), xf);
#pragma unroll
            for (int e = 0; e < 16; e++) acc[m] = __builtin_fmaf(xf[e], wf[e], acc[m]);
        }
    };
    // (a turn's pieces are requested together, in front of the turn before's products: loaded row by row, 15 x 9152 x 272 took 37 us)
    const int pieces = (int)(a.K / 16);
    if (tid < pieces) {
        Pieces now, next;
        fetch(now, tid);
        for (int p = tid; p < pieces; p += 256) {
            fetch(next, p + 256 < pieces ? p + 256 : p);
            __builtin_amdgcn_sched_barrier(0);
            multiply(now);
            now = next;
        }
    }
#pragma unroll
    for (int m = 0; m < ROWS; m++) {
        float v = acc[m];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
        if (lane == 0) red[wave][m] = v;
    }
    __syncthreads();
    if (tid < a.M) {
        float v = ((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid];
        if (a.bias) v = v + ((const float*)a.bias)[n];
        store_f32_as(a.out, a.out_dtype, (int64_t)tid * a.N + n, v);
    }
}
bool mxfp8_few_outputs(const OpsnnQmmArgs& a)
{
    return a.x1_dtype == DT_E4M3 && a.x2_dtype == DT_E4M3 && a.force_variant == 0 && a.batch == 1 && a.N >= 256 && a.M * a.N < 64 * 64 && a.K % 128 == 64;
}
// (`a` as mx_call_ok has passed it, x2 K-contiguous)
static int launch_mxfp8_few_outputs(const OpsnnQmmArgs& a, hipStream_t st)
{
    if (((uintptr_t)a.x2.ptr | (uint64_t)a.x2.col_stride) % 16 || a.x2_scale_mat.col_stride != 2) return OPSNN_NOT_TAKEN;
    note_route("mxfp8_few_outputs");
    const dim3 grid((unsigned)a.N), block(256);
    if (a.M == 1) hipLaunchKernelGGL(mxfp8_few_outputs_kernel<1>, grid, block, 0, st, a);
    else if (a.M == 2) hipLaunchKernelGGL(mxfp8_few_outputs_kernel<2>, grid, block, 0, st, a);
    else if (a.M == 3) hipLaunchKernelGGL(mxfp8_few_outputs_kernel<3>, grid, block, 0, st, a);
    else if (a.M == 4) hipLaunchKernelGGL(mxfp8_few_outputs_kernel<4>, grid, block, 0, st, a);
    else if (a.M <= 8) hipLaunchKernelGGL(mxfp8_few_outputs_kernel<8>, grid, block, 0, st, a);
    else hipLaunchKernelGGL(mxfp8_few_outputs_kernel<16>, grid, block, 0, st, a);   // (fewer than 64 x 64 outputs and 256 columns: 15 rows at most)
    return (int)hipGetLastError();
}

bool mxfp4_rows_wanted(const OpsnnQmmArgs& a);   // qmm_mxfp4_rows.hip
int launch_mxfp4_rows(const OpsnnQmmArgs& a, hipStream_t st);
int launch_fp8_stream(const OpsnnQmmArgs& a, Fp8xForm form, SplitK sk, hipStream_t st);   // qmm_fp8_stream.hip
// What every matrix-core route of this file needs of the call, whatever x2's layout and K's tail: checked before any
// pre-step is launched or a cache entry made.
static bool mx_call_ok(const OpsnnQmmArgs& a)
{
    const bool fp4 = a.x1_dtype == DT_E2M1 && a.x2_dtype == DT_E2M1, fp8 = a.x1_dtype == DT_E4M3 && a.x2_dtype == DT_E4M3;
    const bool a8w4 = a.x1_dtype == DT_E4M3 && a.x2_dtype == DT_E2M1;
    if (!fp4 && !fp8 && !a8w4) return false;
    if (a8w4) {   // launch_mx_a8w4_mfma (qmm_fp8_block.hip): a tile kernel, and a streaming kernel for up to 16 rows
        if (a.out_dtype != DT_BF16 && a.out_dtype != DT_F16) return false;
        if (a.bias && a.bias_dtype != DT_F32 && a.bias_dtype != DT_BF16 && a.bias_dtype != DT_F16) return false;
        if (a.K % 32 != 0 || a.x1.col_stride != 1 || a.x1_scale_mat.col_stride != 2) return false;
        const bool few_rows = a.M <= 32 && a.N >= 256 && a.batch == 1;
        if (!few_rows && a.M * a.N < 64 * 64) return false;
        return (((uintptr_t)a.x1.ptr | (uint64_t)a.x1.row_stride | (uint64_t)a.x1.batch_stride) % 16) == 0;
    }
    if (a.out_dtype != DT_BF16 && a.out_dtype != DT_F16 && a.out_dtype != DT_F32) return false;
    if (a.bias && a.bias_dtype != DT_F32) return false;
    // (fewer than 64 x 64 outputs: only MXFP8's few-rows streams over x2, which want 256 columns and whole half tiles of K: on one thread
    // per output 3 x 15168 x 1088 took 12.4 ms, 16 us here)
    if (a.K % 32 != 0 || (a.M * a.N < 64 * 64 && !(fp8 && a.M <= 32 && a.N >= 256 && a.batch == 1 && a.K % 64 == 0) && !mxfp4_rows_wanted(a))) return false;
    const int64_t ks = (a.K + 63) / 64, epb = fp4 ? 2 : 1;
    if (a.x1.col_stride != 1 || a.x1_scale_mat.col_stride != 2 || a.x1_scale_mat.row_stride != ks * 2) return false;
    if (((uintptr_t)a.x1.ptr | (uint64_t)(a.x1.row_stride / epb) | (uint64_t)(a.x1.batch_stride / epb)) % 16) return false;
    if (a.K % 128 == 0 && ((uintptr_t)a.x1_scale_mat.ptr | (uint64_t)a.x1_scale_mat.row_stride | (uint64_t)a.x1_scale_mat.batch_stride) % 4) return false;
    return true;
}

// Bytes behind the exact route's tables: the K-contiguous copies of an N-contiguous x2, then the padded copies of a K tail.
static uint64_t mx_rest_bytes(const OpsnnQmmArgs& a0)
{
    if (a0.force_variant == OPSNN_VARIANT_PLAIN || opsnn_force_plain() || !mx_call_ok(a0)) return 0;
    OpsnnQmmArgs a = a0;
    uint64_t total = 0;
    MxRelayout R;
    if (mx_relayout_layout(a, R)) {
        total = align_up(R.bytes, 256);
        mx_relayout_view(a, R, (char*)(uintptr_t)256);   // any aligned address: only the layout matters below
    }
    MxPad L;
    if (mx_pad_layout(a, L)) total += L.total;   // (few rows of fp4 leave it unused: the size stays what it always was)
    return total;
}

// Workspace of an MX call: in front, what the exact route of MXFP8 needs (nothing for the other operand pairs), then the
// re-laid-out and padded operand copies.
uint64_t mx_workspace_bytes(const OpsnnQmmArgs& a)
{
    const bool matrix_cores = a.force_variant != OPSNN_VARIANT_PLAIN && !opsnn_force_plain();
    return (matrix_cores ? mx_exact_bytes(a) : 0) + mx_rest_bytes(a);
}

void* weight_cache_blob(const void* src, const void* src2, int64_t K, int64_t N, int bits, int64_t nb, uint64_t bytes, hipStream_t st, bool* fresh);
void weight_cache_commit(void* buffer, hipStream_t st);   // weight_cache.hip
void weight_cache_abandon(void* buffer);
int launch_mxfp8_mfma(const OpsnnQmmArgs& a, hipStream_t st);   // qmm_fp8_block.hip
int launch_mx_a8w4_mfma(const OpsnnQmmArgs& a, hipStream_t st, SplitK sk);   // qmm_fp8_block.hip
int launch_mxfp8_decode(const OpsnnQmmArgs& a, hipStream_t st, SplitK sk);   // qmm_fp8_decode.hip

int launch_mx_mfma(const OpsnnQmmArgs& a0, hipStream_t st, SplitK sk)
{
    if (!mx_call_ok(a0)) return OPSNN_NOT_TAKEN;
    OpsnnQmmArgs a = a0;
    const bool fp4 = a.x1_dtype == DT_E2M1 && a.x2_dtype == DT_E2M1;
    const bool fp8 = a.x1_dtype == DT_E4M3 && a.x2_dtype == DT_E4M3;
    // MXFP8 runs on exact products by default (with two 8-bit operands the scaled matrix instruction aligns its products in
    // a window narrower than fp32: measured on 4096 x 8192 x 8192 with scale exponents in [-4, 4], 1 % of the bf16 outputs
    // one ulp off and the largest relative error above 2^-7); opsnnSetFp8Fast(1) asks for the 8-bit instruction.  With a 4-bit x2 the same instruction is as close to the fp32 sums as
    // exact products are (measured on the same shapes), so that mode keeps it.
    if (const uint64_t front = mx_exact_bytes(a0); front && a.workspace) a.workspace = (char*)a.workspace + front;
    const bool exact = !opsnnGetFp8Fast();

    // Pre-steps, planned in full before the first of them is launched: an N-contiguous x2 is re-laid out K-contiguous (into
    // the weight cache's buffer for this operand when the cache is on -- a hit skips the passes -- else into the workspace);
    // a K tail (K % 128 == 64) then continues on zero-padded copies of all four operands.
    MxRelayout R;
    const bool relayout = mx_relayout_layout(a, R);
    if (!relayout && a.x2.row_stride != 1) return OPSNN_NOT_TAKEN;
    OpsnnQmmArgs planned = a;
    if (relayout) mx_relayout_view(planned, R, (char*)(uintptr_t)256);
    MxPad L;
    // few rows: the kernels that take a K tail as it is.  With the 8-bit instruction asked for too, but for shapes whose 8-bit tiles fill half
    // the CUs and are as fast with x2 from memory, faster from the last-level cache (51 x 3328 x 18624 29.0 and 21.0 us, stream 29.4 and 27.3;
    // 56 x 2944 x 11264 24.7 and 17.9, 19.4 and 18.4; 64 x 5888 x 12288 49 and 35, 32 and 29)
    const bool stream8 = exact || a.M <= 32 || (a.M <= 128 && (a.N <= 16384 || a.K % 128 != 0));
    Fp8StreamPlan spl;
    const bool rows4 = fp4 && mxfp4_rows_wanted(a), few_outputs = mxfp8_few_outputs(a);
    const bool rows8 = fp8 && !few_outputs && stream8 && fp8_stream_plan(a, FP8X_MX, true, spl);
    const bool pad = !rows4 && !rows8 && mx_pad_layout(planned, L);
    if (!pad && !rows4 && !rows8 && !few_outputs && planned.K % 128 != 0) return OPSNN_NOT_TAKEN;
    if (planned.x2_scale_mat.col_stride != 2 || (fp4 || fp8 ? planned.x2_scale_mat.row_stride != (planned.K + 63) / 64 * 2 : planned.x2_scale_mat.row_stride % 4 != 0)) return OPSNN_NOT_TAKEN;
    if (pad && (!a.workspace || (uintptr_t)a.workspace % 16)) return OPSNN_NOT_TAKEN;
    if (relayout) {
        bool fresh = false;
        char* w = (char*)weight_cache_blob(a.x2.ptr, a.x2_scale_mat.ptr, a.K, a.N, a.x2_dtype == DT_E2M1 ? 4 : 8, R.nb * 16 + R.snb, R.bytes, st, &fresh);
        const bool cached = w != nullptr;
        if (!cached) {
            if (!a.workspace || (uintptr_t)a.workspace % 16) return OPSNN_NOT_TAKEN;
            w = (char*)a.workspace;
            a.workspace = w + align_up(R.bytes, 256);
        }
        if (!cached || fresh) {
            const int rc = mx_relayout_run(a, R, w, st);
            if (rc != 0) {
                if (cached) weight_cache_abandon(w);
                return rc;
            }
        }
        if (cached && fresh) weight_cache_commit(w, st);
        mx_relayout_view(a, R, w);
    }
    if (rows4) return launch_mxfp4_rows(a, st);
    if (few_outputs) return launch_mxfp8_few_outputs(a, st);
    if (rows8) {
        const int rc = launch_fp8_stream(a, FP8X_MX, sk, st);
        if (rc != OPSNN_NOT_TAKEN || a.K % 128 != 0) return rc;   // (a K tail was left as it is)
        sk = SplitK{};
    }
    const bool small = a.M <= 128 || a.N <= 128;
    // (the plan that the partial sums were laid out for, or, where a call comes without them, one that leaves K in one piece)
    Mxfp4Plan fp4_plan = mxfp4_tile_plan(a.M, a.N, a.K, a.batch, a.force_variant == 0);
    if (fp4_plan.splits > 1 && (!sk.part || sk.splits != fp4_plan.splits)) fp4_plan = mxfp4_tile_plan(a.M, a.N, a.K, a.batch, false);
    const bool fp4_small = a.force_variant == OPSNN_VARIANT_MX_128 || fp4_plan.small, fp4_cut = fp4_plan.splits > 1 && a.force_variant == 0;
    if (pad) {
        if (!mx_pad_layout(a, L)) return OPSNN_NOT_TAKEN;   // (the same answer as for the planned view: its conditions do not look at x2's address beyond its alignment)
        // (large fp4 tiles in segments deal whole tiles of 128 elements: their operands are padded like everybody's)
        const int rc = fp4 && !fp4_small && !fp4_cut ? mx_pad_scales(a, L, st) : mx_pad_prestep(a, L, st);
        if (rc != 0) return rc;
    }
    if (a.x1_dtype == DT_E4M3 && a.x2_dtype == DT_E2M1) return launch_mx_a8w4_mfma(a, st, sk);   // fp8 x fp4: qmm_fp8_block.hip
    if (fp8 && a.M <= 16) {   // MXFP8 with up to 16 rows: the stream over x2 with x1 in registers (exact products)
        const int rc = launch_mxfp8_decode(a, st, sk);
        if (rc != OPSNN_NOT_TAKEN) return rc;
        if (a.M * a.N < 64 * 64) return OPSNN_NOT_TAKEN;
        sk = SplitK{};   // (the partial sums were laid out for the kernel above; the tile kernels run unsplit)
    }
    // MXFP8 runs on the block kernel of qmm_fp8_block.hip in MX mode (16x16x128 instructions, 64 x 128 per wave, the
    // pipeline tuned for the fp8 block-scale path); the 32x32x64 tile kernel stays available on request
    // (OPSNN_VARIANT_MX_FP8_MFMA) for comparison.  The 8-bit forms of the matrix instruction sum their products with a
    // reduced-width aligner (measured: mean error 1e-5 of sum|terms| per instruction); fp4 products are exact in that
    // datapath.
    const int64_t ks = a.K / 64;  // scale pairs per row
    const int64_t epb = fp4 ? 2 : 1;  // elements per byte

    QgemmParams g{};
    g.a = (const int8_t*)a.x1.ptr; g.b = (const int8_t*)a.x2.ptr;
    g.lda = a.x1.row_stride / epb; g.ldb = a.x2.col_stride / epb;
    g.a_bs = a.x1.batch_stride / epb; g.b_bs = a.x2.batch_stride / epb;
    g.out = a.out; g.M = a.M; g.N = a.N; g.ldc = a.N; g.KB = a.K / epb;
    g.bias = a.bias; g.bias_dt = a.bias_dtype; g.bias_bs = a.bias_batch_stride;
    g.sa = (const uint8_t*)a.x1_scale_mat.ptr; g.sb = (const uint8_t*)a.x2_scale_mat.ptr;
    g.sa_rs = a.x1_scale_mat.row_stride; g.sb_rs = a.x2_scale_mat.row_stride;
    g.sa_bs = a.x1_scale_mat.batch_stride; g.sb_bs = a.x2_scale_mat.batch_stride;
    if (((uintptr_t)g.a | (uintptr_t)g.b | (uint64_t)g.lda | (uint64_t)g.ldb | (uint64_t)g.a_bs | (uint64_t)g.b_bs) % 16) return OPSNN_NOT_TAKEN;
    if (((uintptr_t)g.sa | (uintptr_t)g.sb | (uint64_t)g.sa_rs | (uint64_t)g.sb_rs | (uint64_t)g.sa_bs | (uint64_t)g.sb_bs) % 4) return OPSNN_NOT_TAKEN;
    if (fp8 && exact && a.force_variant != OPSNN_VARIANT_MX_FP8_MFMA && a.force_variant != OPSNN_VARIANT_MX_128) {
        const int rc = launch_mx_exact(a, st, sk);
        if (rc != OPSNN_NOT_TAKEN) return rc;
    }
    if (fp4) {
        // few tiles against a long K: K split over workgroups (fp32 partial sums in front of the workspace), on the tiles
        // chosen below, whole ones
        const bool split = fp4_cut;
        if (split) { g.splits = sk.splits; g.part = (int32_t*)sk.part; }
        // Small tiles: eight waves of 64 x 32 where a CU has at most two workgroups of at most 18 K tiles of 128 each, in one piece, which are a matter of
        // latency (235 x 1536 x 7335 9.5 -> 8.1 us, 8 x 93 x 1152 x 1208 8.7 -> 7.2; 33 drawn calls 0.88 of the time); four of 64 x 64, with fewer reads,
        // where there is more (8 x 36 x 3840 x 10048 50.5 so, 55.5 on eight) and in segments, which end in stores of partial sums (45 drawn calls
        // of such a size 1.017 times as long on eight: 107 x 16896 x 1536 in twelve 16.7 and 17.6, 74 x 9216 x 3840 in six 16.0 and 17.0).
        const bool eight = fp4_small && !split && a.K <= 18 * 128 && (a.M + 127) / 128 * ((a.N + 127) / 128) * a.batch <= 512;
        note_route(eight ? "mxfp4_tiles_128_w8" : fp4_small ? "mxfp4_tiles_128" : "mxfp4_tiles_256", split ? sk.splits : 1);
        if (fp4_small) {
            if (eight) return qgemm_launch<MODE_MXFP4, 128, 128, 64, 2, 4, 4, 1>(g, a.batch, a.out_dtype, st);
            if (split) return qgemm_launch_split_mx<MODE_MXFP4, 128, 128, 64, 2, 2, 4, 1>(g, a.batch, a.out_dtype, st);
            return qgemm_launch<MODE_MXFP4, 128, 128, 64, 2, 2, 4, 1>(g, a.batch, a.out_dtype, st);
        }
        // K tiles of 128 bytes (256 elements) with the scales of two tiles per 16-byte copy; a K that is no whole pair of tiles ends in
        // zeros from the kernel's own page.  (Against 64-byte tiles, on which such a K ran: 2 x 1864 x 1408 x 13208 94 -> 85 us,
        // 4 x 1828 x 3840 x 11712 284 -> 229, 2048 x 8064 x 14336 189 -> 150.)  The K split deals whole pairs.
        if (split && a.K % 512 != 0) return qgemm_launch_split_mx<MODE_MXFP4, 256, 256, 64, 2, 2, 4, 1>(g, a.batch, a.out_dtype, st);
        if (split) return qgemm_launch_split_mx<MODE_MXFP4, 256, 256, 128, 2, 4, 2, 1>(g, a.batch, a.out_dtype, st);
        return qgemm_launch<MODE_MXFP4, 256, 256, 128, 2, 4, 2, 1>(g, a.batch, a.out_dtype, st);
    }
    // FLOAT output: the tile kernel, whose epilogue stores fp32 straight from the registers
    if (a.out_dtype == DT_F32 || a.force_variant == OPSNN_VARIANT_MX_FP8_MFMA || a.force_variant == OPSNN_VARIANT_MX_128) {   // (also the chained-K variants of the tests)
        if (small || a.force_variant == OPSNN_VARIANT_MX_128) return qgemm_launch<MODE_MXFP8, 128, 128, 128, 2, 2, 2, 1>(g, a.batch, a.out_dtype, st);
        return qgemm_launch<MODE_MXFP8, 256, 256, 128, 2, 2, 2, 1>(g, a.batch, a.out_dtype, st);
    }
    // few rows: the 128 x 128 tiles of the tile kernel (the block kernel's 128 x 256 tiles leave most CUs' matrix work on
    // rows that do not exist and half as many workgroups to stream x2)
    if (a.M <= 256) return qgemm_launch<MODE_MXFP8, 128, 128, 128, 2, 2, 2, 1>(g, a.batch, a.out_dtype, st);
    return launch_mxfp8_mfma(a, st);
}

}  // namespace opsnn
