// flash_f32.hip — image-encoder attention on f32 rows, in f32 on the matrix
// cores (v_mfma_f32_16x16x4_f32: f32 operands, products and sums, no
// binary16 or reduced-precision step anywhere).
//
// session::execute(op_self_attention) (S/graph/session.hpp:409-449) with
// self_attend_head's math (S/kernels/attention.hpp:460-486): out_i =
// sum_j softmax_j(scale q_i . k_j) v_j over the n rows of one image.
//
// A block (4 waves) owns 16 query rows of one (image, head); wave w takes a
// quarter of the keys, 32 at a time, with an online softmax, and the four
// partial (max, sum, O) meet in LDS at the end. Per 16 keys a wave computes
//   S^T (16 keys x 16 queries) = K (16 x hd) . q^T      hd/4 products
//   O^T (16 dims x 16 queries) += V^T (16 x 4 keys) . P^T   4 products per 16 dims
// Operands come straight from memory into registers: a 16-byte load of a K
// row is the operand of four products (dims 16u + 4G + i for lane group G and
// product i), a 16-byte load of a V row of four more (O^T tile i holds dims
// 4c + i), and the S^T accumulators are, as they stand, the P^T operand. So
// no LDS is touched before the merge. K of the next 32 keys is loaded while
// the softmax and the output products run, V while the score products run.
//
// What bounds it: the f32 matrix rate (256 FLOP/clk/CU, 4 hd n^2 per head and
// image). One image of 1024 rows, 12 heads of 64: 41.3 us a call (78 TFLOP/s;
// the f32 matrix peak is 157), 1924 us with the row-per-wave kernel; error
// against 64 bits 4.1e-7 (6.4e-7 before). The split into 16-row blocks is for the small case: one 1024-row
// image of 12 heads is 768 blocks, three per CU, all resident at once. Blocks of one
// head are dealt to one XCD, whose L2 then holds that head's K and V.
// Exponentials are expf of the f32 difference to the running max, and
// their sum is kept in double per lane, as in the row-per-wave kernel
// (generic.hip) that this replaces for head sizes in whole 16-byte chunks,
// tiny calls apart (self_f32_mfma_takes).

#include "kernels.hpp"

namespace syn {

namespace {

constexpr uint32_t sf_q = 16;      // query rows per block
constexpr uint32_t sf_waves = 4;
constexpr uint32_t sf_step = 32;   // keys per wave and step

__device__ __forceinline__ f4 sf_mfma(float a, float b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f4 sf_load4(rsrc r, uint32_t off) {
    return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
typedef unsigned int u2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ f2 sf_load2(rsrc r, uint32_t off) {
    return __builtin_bit_cast(f2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
__device__ __forceinline__ float sf_load1(rsrc r, uint32_t off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}

// HDP: head size rounded up to a multiple of 16 (dims past hd read as zeros).
template <int HDP>
__global__ __launch_bounds__(256, HDP <= 80 ? 3 : (HDP <= 128 ? 2 : 1)) void self_f32_mfma_kernel(const flash_args a,
                                                                                              uint32_t tiles) {
    constexpr int NU = HDP / 16;            // 16-dim units: K chunks per key and lane, O^T tiles
    constexpr int N4 = HDP / 64;            // V: 64-dim groups (16-byte loads, 4 tiles),
    constexpr int N2 = HDP % 64 / 32;       //    then at most one 32-dim group (8-byte, 2 tiles)
    constexpr int N1 = HDP % 32 / 16;       //    and one 16-dim group (4-byte, 1 tile)
    constexpr int E = sf_step / 16;         // 16-key tiles per step
    constexpr uint32_t OROW = HDP + 4;      // LDS row of a query's partial output
    __shared__ __attribute__((aligned(16))) float lo[sf_waves][sf_q][OROW];
    __shared__ float lm[sf_waves][sf_q];
    __shared__ double ls[sf_waves][sf_q];

    const uint32_t tid = threadIdx.x;
    const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t ln = tid & 63, G = ln >> 4, c = ln & 15;
    const uint32_t n = a.n, hd = a.hd;
    // Blocks go to the 8 XCDs in turn; each XCD takes a contiguous run of
    // (image, head, query tile), so a head's blocks share an L2.
    const uint32_t total = gridDim.x, xcd = blockIdx.x % 8;
    const uint32_t id = xcd * (total / 8) + min(xcd, total % 8) + blockIdx.x / 8;
    const uint32_t unit = id / tiles, q0 = id % tiles * sf_q;
    const uint32_t h = unit % a.n_heads, img = unit / a.n_heads;
    const std::size_t base = static_cast<std::size_t>(img) * n * a.row + static_cast<std::size_t>(h) * hd;
    const uint32_t bytes = n * a.row * 4 - h * hd * 4;  // to the image's end
    const rsrc qr = make_rsrc(static_cast<const float*>(a.q) + base, bytes);
    const rsrc kr = make_rsrc(static_cast<const float*>(a.k_rows) + base, bytes);
    const rsrc vr = make_rsrc(static_cast<const float*>(a.v_rows) + base, bytes);
    const uint32_t row4 = a.row * 4;

    // This wave's keys: a quarter, in whole 16-key tiles.
    const uint32_t per = ((n + 15) / 16 + sf_waves - 1) / sf_waves * 16;
    const uint32_t k_begin = min(w * per, n), k_end = min(k_begin + per, n);

    // Keys of row tile e: the A operand's row c is key t + 16 e + c. Rows past
    // k_end read zeros (they are masked below).
    f4 kb[E][NU], vb4[E][4][N4 > 0 ? N4 : 1];
    f2 vb2[E][4];
    float vb1[E][4];
    const auto load_k = [&](uint32_t t) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const uint32_t key = t + 16 * e + c;
            const uint32_t off = key < k_end ? key * row4 + 16 * G : buffer_oob;
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                kb[e][u] = sf_load4(kr, 16 * u + 4 * G < hd ? off + 64 * u : buffer_oob);
            }
        }
    };
    // V of key t + 16 e + 4 G + i (the key that register i of S^T tile e holds).
    const auto load_v = [&](uint32_t t) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t key = t + 16 * e + 4 * G + i;
                const uint32_t off = key < k_end ? key * row4 : buffer_oob;
#pragma unroll
                for (int j = 0; j < N4; ++j) {
                    vb4[e][i][j] = sf_load4(vr, 64 * j + 4 * c < hd ? off + 256 * j + 16 * c : buffer_oob);
                }
                if constexpr (N2 > 0) {
                    vb2[e][i] = sf_load2(vr, 64 * N4 + 2 * c < hd ? off + 256 * N4 + 8 * c : buffer_oob);
                }
                if constexpr (N1 > 0) {
                    constexpr uint32_t d1 = 64 * N4 + 32 * N2;
                    vb1[e][i] = sf_load1(vr, d1 + c < hd ? off + 4 * d1 + 4 * c : buffer_oob);
                }
            }
        }
    };

    if (k_begin < k_end) {
        load_k(k_begin);
    }
    f4 qv[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        qv[u] = sf_load4(qr, q0 + c < n && 16 * u + 4 * G < hd ? (q0 + c) * row4 + 64 * u + 16 * G : buffer_oob);
    }

    f4 o[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        o[u] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    float m_run = -INFINITY;  // query c's running max over this wave's keys
    double l_run = 0.0;       // this lane's share of its sum
    for (uint32_t t = k_begin; t < k_end; t += sf_step) {
        load_v(t);
        f4 s[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            s[e] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (int u = 0; u < NU; ++u) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    s[e] = sf_mfma(kb[e][u][i], qv[u][i], s[e]);
                }
            }
        }
        load_k(t + sf_step);  // (past k_end: zeros, no request)
        float mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < E; ++e) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float x = s[e][i] * a.scale;
                s[e][i] = t + 16 * e + 4 * G + i < k_end ? x : -INFINITY;
                mx = fmaxf(mx, s[e][i]);
            }
        }
        mx = max32(max16(mx));
        const bool grow = mx > m_run;
        if (__builtin_amdgcn_ballot_w64(grow) != 0) {
            // A query whose max did not move is scaled by 1.
            const float m_new = grow ? mx : m_run;
            const float alpha = grow ? expf(m_run - m_new) : 1.0f;
            m_run = m_new;
            l_run *= static_cast<double>(alpha);
#pragma unroll
            for (int u = 0; u < NU; ++u) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    o[u][i] *= alpha;
                }
            }
        }
        const float m_use = m_run == -INFINITY ? 0.0f : m_run;  // no finite score yet: every term is exp(-inf)
#pragma unroll
        for (int e = 0; e < E; ++e) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[e][i] = expf(s[e][i] - m_use);
                l_run += static_cast<double>(s[e][i]);
            }
        }
        // O^T tile (64-dim group j, i): dims 64 j + 4 c' + i; the 32- and
        // 16-dim groups likewise with their width.
#pragma unroll
        for (int e = 0; e < E; ++e) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int j = 0; j < N4; ++j) {
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        o[4 * j + x] = sf_mfma(vb4[e][i][j][x], s[e][i], o[4 * j + x]);
                    }
                }
                if constexpr (N2 > 0) {
                    o[4 * N4] = sf_mfma(vb2[e][i][0], s[e][i], o[4 * N4]);
                    o[4 * N4 + 1] = sf_mfma(vb2[e][i][1], s[e][i], o[4 * N4 + 1]);
                }
                if constexpr (N1 > 0) {
                    o[NU - 1] = sf_mfma(vb1[e][i], s[e][i], o[NU - 1]);
                }
            }
        }
    }

    // ---- merge the four waves' partials ----
    l_run += __shfl_xor(l_run, 16, wave);
    l_run += __shfl_xor(l_run, 32, wave);
    if (G == 0) {
        lm[w][c] = m_run;
        ls[w][c] = l_run;
    }
    // Lane (G, c), register r of a tile: query c, tile row 4 G + r.
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const uint32_t tr = 4 * G + r;
#pragma unroll
        for (int j = 0; j < N4; ++j) {
            *reinterpret_cast<f4*>(&lo[w][c][64 * j + 4 * tr]) =
                f4{o[4 * j][r], o[4 * j + 1][r], o[4 * j + 2][r], o[4 * j + 3][r]};
        }
        if constexpr (N2 > 0) {
            *reinterpret_cast<f2*>(&lo[w][c][64 * N4 + 2 * tr]) = f2{o[4 * N4][r], o[4 * N4 + 1][r]};
        }
        if constexpr (N1 > 0) {
            lo[w][c][64 * N4 + 32 * N2 + tr] = o[NU - 1][r];
        }
    }
    __syncthreads();
    for (uint32_t x = tid; x < sf_q * (HDP / 4); x += 256) {
        const uint32_t q = x / (HDP / 4), d = x % (HDP / 4) * 4;
        if (q0 + q >= n || d >= hd) {
            continue;
        }
        float m = lm[0][q];
#pragma unroll
        for (uint32_t v = 1; v < sf_waves; ++v) {
            m = fmaxf(m, lm[v][q]);
        }
        f4 r = f4{0.0f, 0.0f, 0.0f, 0.0f};
        double l = 0.0;
#pragma unroll
        for (uint32_t v = 0; v < sf_waves; ++v) {
            const float mv = lm[v][q];
            const float f = mv == -INFINITY ? 1.0f : expf(mv - m);  // (a wave with no finite score: its sums are 0 or NaN)
            const f4 p = *reinterpret_cast<const f4*>(&lo[v][q][d]);
            l += ls[v][q] * static_cast<double>(f);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                r[i] = fmaf(p[i], f, r[i]);
            }
        }
        const auto inv = static_cast<float>(1.0 / l);
        float* out = a.out + base + static_cast<std::size_t>(q0 + q) * a.row + d;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            r[i] *= inv;
        }
        *reinterpret_cast<f4*>(out) = r;
    }
}

template <int HDP>
hipError_t launch_hd(const flash_args& a, hipStream_t stream) {
    const uint32_t tiles = (a.n + sf_q - 1) / sf_q;
    self_f32_mfma_kernel<HDP><<<tiles * a.n_heads * a.batch, 256, 0, stream>>>(a, tiles);
    return hipGetLastError();
}

}  // namespace

bool self_f32_mfma_takes(const flash_args& a) {
    // Rows are read and written 16 bytes at a time (heads of whole 8-dim
    // chunks are aligned by the interface, those of 4, 12, ... dims need not
    // be); a launch takes fewer than 2^32 threads in one dimension.
    const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const bool fits = a.hd % 4 == 0 && aligned(a.q) && aligned(a.k_rows) && aligned(a.v_rows) && aligned(a.out) &&
                      uint64_t{a.n} * a.row * 4 < (uint64_t{1} << 31) &&
                      (uint64_t{a.n} + sf_q - 1) / sf_q * a.n_heads * a.batch < (uint64_t{1} << 24);
    // A few short rows of tiny heads are done by a wave a row before this
    // kernel's merge is: us in a graph, row per wave against this one, one
    // head: 4 dims 1 row 2.4 / 3.1, 32 rows 3.3 / 3.4; 8 dims 8 rows 2.8 /
    // 3.1, 16 rows 3.1 / 3.2, 32 rows 3.6 / 3.3; 12 dims 8 rows 3.1 / 3.1; 16
    // dims 2 rows 3.2 / 3.2; and while the rows are few: 8 dims, 16 rows, 64
    // images 3.5 / 3.5, of 12 heads 8.3 / 3.9.
    const bool tiny = a.hd <= 12 && uint64_t{a.hd} * a.n <= 160 && uint64_t{a.n} * a.n_heads * a.batch <= 1536;
    return fits && !tiny;
}

hipError_t launch_self_f32_mfma(const flash_args& a, hipStream_t stream) {
    const uint32_t hd = a.hd;
    if (hd <= 32) {
        return launch_hd<32>(a, stream);
    }
    if (hd <= 64) {
        return launch_hd<64>(a, stream);
    }
    if (hd <= 80) {
        return launch_hd<80>(a, stream);
    }
    if (hd <= 96) {
        return launch_hd<96>(a, stream);
    }
    if (hd <= 128) {
        return launch_hd<128>(a, stream);
    }
    if (hd <= 192) {
        return launch_hd<192>(a, stream);
    }
    return launch_hd<256>(a, stream);
}

}  // namespace syn
