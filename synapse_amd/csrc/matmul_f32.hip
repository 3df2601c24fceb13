// matmul_f32.hip — products with F32 weights: out[r][o] = sum_c w[o][c]
// x[r][c] (+ bias[o]) (session::execute(op_matmul), S/graph/session.hpp:
// 287-302; op_add_bias, :306-312), f32 operands, products and sums.
//
// Two kernels, by the number of activation rows (matmul_f32_plan.hpp):
// - gemv_f32_kernel, few rows (a decode step): bound by reading w once. One
//   wave per weight row, 16 loads in flight; up to four activation rows share
//   a pass over w.
// - gemm_f32_kernel, many rows (an image's patches, a prompt): bound by the
//   f32 matrix cores. Tiles through LDS, v_mfma_f32_32x32x2_f32.

#include "kernels.hpp"
#include "matmul_f32_plan.hpp"

namespace syn {

namespace {

// Sum over the wave by lane xor 32, 16, 8, 4, 2, 1, the same in every lane, on
// the VALU: swaps across the halves and rows, then rotations inside a row
// (after xor 8 the row repeats every 8 lanes, so a rotation by 4 is xor 4).
__device__ __forceinline__ float mf_wave_sum(float v) {
    v = sum16(sum32(v));
    v += dpp_read<0x128>(v);  // row_ror:8
    v += dpp_read<0x124>(v);  // row_ror:4
    v += dpp_read<dpp_quad_xor2>(v);
    v += dpp_read<dpp_quad_xor1>(v);
    return v;
}

// ---- few activation rows ----------------------------------------------------------
//
// Lane l takes columns l, l + 64, ... in order, then the lanes are summed
// (mf_wave_sum). One dword per lane and load on purpose: the order of the
// sums decides on which side of a binary16 boundary a later q, k or p falls,
// and this one is held to the reference's logits to 1e-4 by the golden
// models; 16-byte loads would take another. What the loads need instead is
// number: 16 weight loads (4 KB) in flight per wave and eight waves per SIMD.
// One row of 16000 x 2048 21.5 us a call (6.1 TB/s), 5632 x 2048 8.0, 2048 x
// 5632 8.5; with one load in flight per lane 39.4, 12.8 and 29.1.
// Row resources end at the row, so columns past it add zeros.
// U loads are in flight per lane: as many as the row has for a lane, at most
// 16 (a load past the row costs its issue all the same: 20000 x 16 with 3
// rows 6.2 us a call, 15.5 with 16 loads whatever the row has; one load at a
// time, one row per pass: 7.2). The order of the sums is the same.
template <int NR, int U>
__global__ __launch_bounds__(256) void gemv_f32_kernel(const float* w, const float* x, const float* bias, float* out,
                                                       uint32_t n, uint32_t rows, uint32_t cols) {
    const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t ln = threadIdx.x & 63;
    const uint32_t o = blockIdx.x * 4 + wv;
    const uint32_t r0 = blockIdx.y * NR;
    if (o >= rows) {
        return;  // wave-uniform
    }
    const auto load = [](rsrc r, uint32_t off) {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
    };
    const rsrc wr = make_rsrc(w + static_cast<std::size_t>(o) * cols, cols * 4);
    rsrc xr[NR];
    float acc[NR];
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        xr[j] = make_rsrc(x + static_cast<std::size_t>(min(r0 + j, n - 1)) * cols, cols * 4);
        acc[j] = 0.0f;
    }
    for (uint32_t c = 0; c < cols * 4; c += 256 * U) {
        float wb[U], xb[NR][U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            wb[u] = load(wr, c + 256 * u + 4 * ln);
        }
#pragma unroll
        for (int j = 0; j < NR; ++j) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                xb[j][u] = load(xr[j], c + 256 * u + 4 * ln);
            }
        }
        __builtin_amdgcn_sched_barrier(0);  // all the loads before the first product
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                acc[j] = fmaf(wb[u], xb[j][u], acc[j]);
            }
        }
    }
    const float bo = bias != nullptr ? bias[o] : 0.0f;
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        const float s = mf_wave_sum(acc[j]);
        if (ln == 0 && r0 + j < n) {
            out[static_cast<std::size_t>(r0 + j) * rows + o] = bias != nullptr ? s + bo : s;
        }
    }
}

// ---- many activation rows ------------------------------------------------------------
//
// A block of 4 waves owns 32 WM activation rows x 32 WN weight rows; wave
// (wm, wn, wk) a 32 x 32 tile of it over every WK-th group of 32 columns. A
// stage of 32 WK columns reaches LDS by direct copies, two stages deep: per
// group of 32 columns a row is 8 chunks of 16 bytes, chunk k in slot
// k ^ (row % 8), so that the operand reads (32 rows, one chunk each per lane
// half) spread over the banks. A lane's chunk feeds four products (columns
// 8 u + 4 H + i for lane half H and product i). A stage's products sum from
// zero in four chains of 8 columns, which are added to one of four running
// sums: short chains instead of one of cols, so that the rounding error stays
// that of one wave per output (gemv_f32_kernel): against 64 bits at 768
// columns 7.0e-8 and 7.1e-8 of the result's norm. (One chain of 32 a stage
// and one running sum: 1.0e-7, and 42.1 us where this takes 45.7.)
//
// Bound by the f32 matrix rate: 1024 rows of 3072 x 768 45.7 us a call (106
// TFLOP/s of 157; 1317 us with one wave per output), 4096 rows 109 TFLOP/s.
template <int WM, int WN, int WK>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* w, const float* x, const float* bias, float* out,
                                                       uint32_t n, uint32_t rows, uint32_t cols, uint32_t row_tiles) {
    static_assert(WM * WN * WK == 4, "four waves");
    constexpr uint32_t BM = 32 * WM, BN = 32 * WN, BR = BM + BN;
    constexpr uint32_t STAGE = BR * WK * 128;
    constexpr int COPIES = STAGE / 4096;  // 1 KB copies per wave and stage
    constexpr uint32_t GROUPS = BR / 8;
    static_assert(GROUPS % 4 == 0 && BM % 32 == 0, "four waves' copies of one operand");
    __shared__ __attribute__((aligned(16))) char lds0[STAGE];
    __shared__ __attribute__((aligned(16))) char lds1[STAGE];

    const uint32_t tid = threadIdx.x;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t ln = tid & 63, H = ln >> 5, c = ln & 31;
    const uint32_t wm = wv % WM, wn = wv / WM % WN, wk = wv / (WM * WN);
    // Blocks go to the 8 XCDs in turn; each XCD takes a contiguous run of
    // tiles, activation tiles fastest, so its L2 holds a band of w and x.
    const uint32_t total = gridDim.x, xcd = blockIdx.x % 8;
    const uint32_t id = xcd * (total / 8) + min(xcd, total % 8) + blockIdx.x / 8;
    const uint32_t t0 = id % row_tiles * BM, o0 = id / row_tiles * BN;
    // Rows past the last read zeros.
    const rsrc xr = make_rsrc(x + static_cast<std::size_t>(t0) * cols, min(BM, n - t0) * cols * 4);
    const rsrc wr = make_rsrc(w + static_cast<std::size_t>(o0) * cols, min(BN, rows - o0) * cols * 4);

    // Copy j = 4 i + wv of a stage: rows 8 (j % GROUPS) .. + 7 (activation
    // rows first, then weight rows) of 32-column group j / GROUPS; lane l row
    // l / 8, slot l % 8. Four groups of 8 rows are of one operand, so which
    // one does not hang on the wave.
    uint32_t off[COPIES], col[COPIES];
#pragma unroll
    for (int i = 0; i < COPIES; ++i) {
        constexpr uint32_t G = GROUPS;
        const uint32_t first = 4 * i % G < BM / 8 ? 4 * i % G : 4 * i % G - BM / 8;
        const uint32_t row = 8 * (first + wv) + ln / 8;
        col[i] = 4 * i / G * 32 + 4 * ((ln & 7) ^ (ln / 8));
        off[i] = (row * cols + col[i]) * 4;
    }
    const auto issue = [&](uint32_t k0, char* stage) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < COPIES; ++i) {
            const uint32_t at = k0 + col[i] < cols ? off[i] + 4 * k0 : buffer_oob;
            buffer_load16_lds(4 * i % GROUPS < BM / 8 ? xr : wr, stage + 4096 * i + 1024 * wv, at);
        }
    };
    const auto landed = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
    };

    f16v sums[4] = {};  // of every fourth stage
    const auto compute = [&](const char* stage, f16v& acc) __attribute__((always_inline)) {
        const char* xs = stage + (wk * BR + 32 * wm + c) * 128;
        const char* ws = stage + (wk * BR + BM + 32 * wn + c) * 128;
        f4 xa[4], wb[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t slot = 16 * ((2 * u + H) ^ (c & 7));  // (32-row groups: row % 8 = c % 8)
            xa[u] = *reinterpret_cast<const f4*>(xs + slot);
            wb[u] = *reinterpret_cast<const f4*>(ws + slot);
        }
        f16v part[4] = {};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                part[u] = __builtin_amdgcn_mfma_f32_32x32x2f32(xa[u][i], wb[u][i], part[u], 0, 0, 0);
            }
        }
        acc += (part[0] + part[1]) + (part[2] + part[3]);
    };
    // Stage s computes from one buffer while stage s + 1 lands in the other.
    // Each wave waits for its own copies, then the barrier: the stage is
    // whole, and every wave is done with the buffer the next copies fill.
    const uint32_t stages = (cols + 32 * WK - 1) / (32 * WK);
    issue(0, lds0);
    for (uint32_t s = 0; s < stages; s += 4) {
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e) {
            if (s + e < stages) {
                landed();
                if (s + e + 1 < stages) {
                    issue((s + e + 1) * 32 * WK, e % 2 == 0 ? lds1 : lds0);
                }
                compute(e % 2 == 0 ? lds0 : lds1, sums[e]);
            }
        }
    }

    f16v acc = (sums[0] + sums[1]) + (sums[2] + sums[3]);
    if constexpr (WK > 1) {
        // The column groups' sums, in order: waves wk > 0 to LDS, wave wk = 0
        // adds them (in double: 588 columns 8.2e-8 against 64 bits, 8.82e-8 in
        // float, 8.80e-8 with one wave per output).
        lds_barrier();
        f4* part = reinterpret_cast<f4*>(lds0);
        if (wk > 0) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                part[((wv - WM * WN) * 4 + q) * 64 + ln] = f4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
            }
        }
        lds_barrier();
        if (wk > 0) {
            return;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            f4 p[WK - 1];
#pragma unroll
            for (int k = 1; k < WK; ++k) {
                p[k - 1] = part[((wv + (k - 1) * WM * WN) * 4 + q) * 64 + ln];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                double s = acc[4 * q + i];
#pragma unroll
                for (int k = 1; k < WK; ++k) {
                    s += static_cast<double>(p[k - 1][i]);
                }
                acc[4 * q + i] = static_cast<float>(s);
            }
        }
    }
    const uint32_t o = o0 + 32 * wn + c;
    if (o < rows) {
        const float bo = bias != nullptr ? bias[o] : 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint32_t r = t0 + 32 * wm + 8 * (i / 4) + 4 * H + i % 4;
            if (r < n) {
                out[static_cast<std::size_t>(r) * rows + o] = bias != nullptr ? acc[i] + bo : acc[i];
            }
        }
    }
}

}  // namespace

hipError_t launch_matmul(const float* w, const float* x, const float* bias, float* out, uint32_t n, uint32_t rows,
                         uint32_t cols, hipStream_t stream) {
    const matmul_f32_plan p = plan_matmul_f32(n, rows, cols);
    if (p.blocks_x == 0) {
        return hipErrorInvalidConfiguration;
    }
    if (p.bm != 0) {
        const auto go = [&](auto kernel) {
            kernel<<<p.blocks_x, 256, 0, stream>>>(w, x, bias, out, n, rows, cols, (n + p.bm - 1) / p.bm);
        };
        if (p.bm == 64) {
            go(gemm_f32_kernel<2, 2, 1>);
        } else if (p.bn == 64) {
            go(gemm_f32_kernel<1, 2, 2>);
        } else {
            go(gemm_f32_kernel<1, 1, 4>);
        }
        return hipGetLastError();
    }
    const uint32_t nr = n >= 4 ? 4 : (n >= 2 ? 2 : 1);
    const dim3 grid(p.blocks_x, p.blocks_y);
    const auto gemv = [&]<int NR>() {
        const auto go = [&](auto kernel) { kernel<<<grid, 256, 0, stream>>>(w, x, bias, out, n, rows, cols); };
        if (cols <= 64) {
            go(gemv_f32_kernel<NR, 1>);
        } else if (cols <= 256) {
            go(gemv_f32_kernel<NR, 4>);
        } else if (cols <= 512) {
            go(gemv_f32_kernel<NR, 8>);
        } else {
            go(gemv_f32_kernel<NR, 16>);
        }
    };
    if (nr == 4) {
        gemv.template operator()<4>();
    } else if (nr == 2) {
        gemv.template operator()<2>();
    } else {
        gemv.template operator()<1>();
    }
    return hipGetLastError();
}

}  // namespace syn
