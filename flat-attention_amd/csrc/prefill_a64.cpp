// Host side of the assembly prefill kernels fa_prefill_a64_bf16 (contiguous K/V) and
// fa_prefill_a64_paged_bf16 (K/V in a pool of 16-row pages through block tables), their f16
// twins fa_prefill_a64_f16 / fa_prefill_a64_paged_f16 and the precise-score
// fa_prefill_a64_precise_bf16, generated by
// gen_prefill_a64.py, assembled into one gfx950 code object and embedded in this library:
// per-device module load and the hipModuleLaunchKernel of one launch. The kernel computes the same prefill as
// prefill_mfma16<bf16> (forward_reference src/lib.rs:454-520 with RoPE rotated_pair
// src/rotary_grouped.rs:37-50 applied to Q), with 64 query rows per wave.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <atomic>
#include <mutex>

#include "kernels.hpp"
#include "prefill_a64_args.h"

namespace fa {

extern const unsigned char kPrefillA64Co[];
extern const size_t kPrefillA64CoSize;

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_mu;
hipModule_t g_mod[kMaxDevices] = {};
hipFunction_t g_fn[kMaxDevices] = {};        // contiguous K/V
hipFunction_t g_fn_paged[kMaxDevices] = {};  // K/V in a pool of 16-row pages
hipFunction_t g_fn_prec[kMaxDevices] = {};   // precise scores (K and Q with their residuals)
hipFunction_t g_fn_f16[kMaxDevices] = {};    // f16 storage, contiguous K/V
hipFunction_t g_fn_paged_f16[kMaxDevices] = {};  // f16 storage, 16-row pages

// Granlund-Montgomery round-up magic of d for n < 2^24: n / d = (mulhi(n, m) + n) >> s.
void fastdiv(uint32_t d, uint32_t* m, uint32_t* s) {
    uint32_t sh = 0;
    while ((1u << sh) < d) ++sh;
    *m = (uint32_t)((((uint64_t)1 << 32) * (((uint64_t)1 << sh) - d)) / d + 1);
    *s = sh;
}

hipFunction_t current_fn(bool paged, bool prec, bool f16) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lock(g_mu);
    if (f16) return prec ? nullptr : paged ? g_fn_paged_f16[dev] : g_fn_f16[dev];
    return paged ? g_fn_paged[dev] : prec ? g_fn_prec[dev] : g_fn[dev];
}

struct Args {
    unsigned char b[FA_A64_ARG_BYTES];
    template <typename T>
    void put(int off, T v) { std::memcpy(b + off, &v, sizeof v); }
};
}  // namespace

hipError_t prefill_a64_load(int device) {
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_fn[device]) return hipSuccess;
    hipModule_t mod = nullptr;
    hipError_t e = hipModuleLoadData(&mod, kPrefillA64Co);
    if (e != hipSuccess) return e;
    hipFunction_t fn = nullptr, fn_paged = nullptr, fn_prec = nullptr, fn_f16 = nullptr,
                  fn_paged_f16 = nullptr;
    e = hipModuleGetFunction(&fn, mod, FA_A64_KERNEL);
    if (e == hipSuccess) e = hipModuleGetFunction(&fn_paged, mod, FA_A64_KERNEL_PAGED);
    if (e == hipSuccess) e = hipModuleGetFunction(&fn_prec, mod, FA_A64_KERNEL_PREC);
    if (e == hipSuccess) e = hipModuleGetFunction(&fn_f16, mod, FA_A64_KERNEL_F16);
    if (e == hipSuccess) e = hipModuleGetFunction(&fn_paged_f16, mod, FA_A64_KERNEL_PAGED_F16);
    if (e != hipSuccess) {
        (void)hipModuleUnload(mod);
        return e;
    }
    g_mod[device] = mod;
    g_fn[device] = fn;
    g_fn_paged[device] = fn_paged;
    g_fn_prec[device] = fn_prec;
    g_fn_f16[device] = fn_f16;
    g_fn_paged_f16[device] = fn_paged_f16;
    return hipSuccess;
}

int device_cus() {
    static std::atomic<int> known[kMaxDevices];
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
    if ((cus = known[dev].load(std::memory_order_relaxed)) > 0) return cus;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0)
        return 256;
    known[dev].store(cus, std::memory_order_relaxed);
    return cus;
}

bool prefill_a64_eligible(Dtype dt, bool paged, const PrefillArgs& a) {
    if (!a.a64 || (dt != Dtype::BF16 && dt != Dtype::F16) || a.head_dim != 128 || a.rope_k ||
        a.split_qk || a.var_meta)
        return false;
    // paged K/V: 16-row pages (one transfer instruction reads one page), block tables whose
    // rows (4-byte entries) the scalar offsets of one sequence address in 32 bits
    if (paged && (a.page_size != 16 || !a.block_tables || a.bt_stride <= 0 ||
                  (uint64_t)a.batch * (uint64_t)a.bt_stride * 4u >= 0x7f000000ull ||
                  (uint64_t)a.k_ss * 2u * 16u >= (1ull << 31)))
        return false;
    const int g = a.group;
    if (g <= 0 || (g & (g - 1)) || g > 256) return false;
    // Q is scaled by scale * log2 e before its one rounding to 16 bits, which only costs nothing
    // when Q is rounded anyway: after its RoPE rotation. Unrotated bf16 Q keeps the HIP kernels
    // (exact products).
    if (!a.rope_q || !a.rope_table || a.rope_rows < a.q_rope_offset + a.q_len) return false;
    // 16-byte aligned rows and bases (every access is 16 bytes wide, or 8 for O)
    const uint64_t al = (uint64_t)(uintptr_t)a.q | (uint64_t)(uintptr_t)a.k |
                        (uint64_t)(uintptr_t)a.v | (uint64_t)(uintptr_t)a.o;
    if (al % 16 || (uint64_t)(uintptr_t)a.lse % 4) return false;
    if (a.q_ss % 8 || a.q_sh % 8 || a.q_sb % 8 || a.k_ss % 8 || a.k_sh % 8 || a.k_sb % 8 ||
        a.o_ss % 4 || a.o_sh % 4 || a.o_sb % 4 || a.k_ss < 128)
        return false;
    // 32-bit offsets within one (batch, kv head) slice, below the resource limit 2^31
    const uint64_t lim = 0x7f000000ull;
    const uint64_t rows = (uint64_t)a.q_len;
    if (!paged && (uint64_t)a.kv_len * (uint64_t)a.k_ss * 2 >= lim) return false;
    if (((uint64_t)(g - 1) * a.q_sh + (rows - 1) * a.q_ss + 128) * 2 >= lim) return false;
    if (((uint64_t)(g - 1) * a.o_sh + (rows - 1) * a.o_ss + 128) * 2 >= lim) return false;
    if (((uint64_t)(g - 1) * a.lse_sh + rows) * 4 >= lim) return false;
    if ((uint64_t)a.q_sh * 2 >= (1ull << 32) || (uint64_t)a.o_sh * 2 >= (1ull << 32) ||
        (uint64_t)a.lse_sh * 4 >= (1ull << 32))
        return false;
    if (a.rope_q && (uint64_t)a.rope_rows * 512 >= lim) return false;
    // precise scores: bf16, contiguous K with its residual 16-byte aligned
    if (a.k_lo && (paged || dt != Dtype::BF16 || (uint64_t)(uintptr_t)a.k_lo % 16)) return false;
    // block indices in 24 bits (SALU fast division)
    const uint64_t nqb = (rows * g + 255) / 256;
    if ((uint64_t)a.batch * a.kv_heads * nqb >= (1u << 24)) return false;
    return current_fn(paged, a.k_lo != nullptr, dt == Dtype::F16) != nullptr;
}

unsigned prefill_a64_workgroups(const PrefillArgs& a) {
    const uint64_t nb = (uint64_t)a.batch * a.kv_heads * (((int64_t)a.q_len * a.group + 255) / 256);
    return (unsigned)std::min<uint64_t>(nb, (uint64_t)device_cus());
}

void launch_prefill_a64(Dtype dt, const PrefillArgs& a, bool paged, hipStream_t s,
                        unsigned grid[3], unsigned* block) {
    int gshift = 0;
    while ((1 << gshift) < a.group) ++gshift;
    const uint32_t nqb = (uint32_t)(((int64_t)a.q_len * a.group + 255) / 256);
    const uint32_t nb = (uint32_t)a.batch * (uint32_t)a.kv_heads * nqb;
    grid[0] = nb;
    grid[1] = grid[2] = 1;
    *block = 256;
    const uint32_t units = (uint32_t)a.batch * (uint32_t)a.kv_heads;
    // persistent grid: one workgroup per CU (each holds a CU's LDS and a SIMD's registers per
    // wave) walking the snake-ordered block list
    const uint32_t wg = prefill_a64_workgroups(a);
    grid[0] = wg;
    Args x{};
    x.put<uint64_t>(FA_A64_OFF_Q, (uint64_t)(uintptr_t)a.q);
    x.put<uint64_t>(FA_A64_OFF_K, (uint64_t)(uintptr_t)a.k);
    x.put<uint64_t>(FA_A64_OFF_V, (uint64_t)(uintptr_t)a.v);
    x.put<uint64_t>(FA_A64_OFF_O, (uint64_t)(uintptr_t)a.o);
    x.put<uint64_t>(FA_A64_OFF_LSE, (uint64_t)(uintptr_t)a.lse);
    x.put<uint64_t>(FA_A64_OFF_ROPE, (uint64_t)(uintptr_t)a.rope_table);
    x.put<uint64_t>(FA_A64_OFF_Q_SB, (uint64_t)a.q_sb * 2);
    if (paged) {
        // the k_sb slot carries the block-table row stride (a page pool has no batch stride)
        x.put<uint64_t>(FA_A64_OFF_BT, (uint64_t)(uintptr_t)a.block_tables);
        x.put<uint32_t>(FA_A64_OFF_BT_STRIDE, (uint32_t)a.bt_stride);
    } else {
        x.put<uint64_t>(FA_A64_OFF_K_SB, (uint64_t)a.k_sb * 2);
        // precise: the residual's distance from K (the block-table slot of the paged kernel)
        if (a.k_lo)
            x.put<uint64_t>(FA_A64_OFF_KLO_OFF,
                            (uint64_t)((uintptr_t)a.k_lo - (uintptr_t)a.k));
    }
    x.put<uint64_t>(FA_A64_OFF_O_SB, (uint64_t)a.o_sb * 2);
    x.put<uint64_t>(FA_A64_OFF_LSE_SB, (uint64_t)a.lse_sb * 4);
    x.put<uint64_t>(FA_A64_OFF_K_SH, (uint64_t)a.k_sh * 2);
    x.put<uint32_t>(FA_A64_OFF_Q_SH, (uint32_t)(a.q_sh * 2));
    x.put<uint32_t>(FA_A64_OFF_O_SH, (uint32_t)(a.o_sh * 2));
    x.put<uint32_t>(FA_A64_OFF_LSE_SH, (uint32_t)(a.lse_sh * 4));
    x.put<uint32_t>(FA_A64_OFF_Q_SS, (uint32_t)(a.q_ss * 2));
    x.put<uint32_t>(FA_A64_OFF_O_SS, (uint32_t)(a.o_ss * 2));
    x.put<uint32_t>(FA_A64_OFF_K_SS, (uint32_t)(a.k_ss * 2));
    x.put<int32_t>(FA_A64_OFF_Q_LEN, a.q_len);
    x.put<int32_t>(FA_A64_OFF_KV_LEN, a.kv_len);
    x.put<int32_t>(FA_A64_OFF_GSHIFT, gshift);
    x.put<int32_t>(FA_A64_OFF_KV_HEADS, a.kv_heads);
    x.put<int32_t>(FA_A64_OFF_CAUSAL, a.causal ? 1 : 0);
    x.put<int32_t>(FA_A64_OFF_CAUSAL_OFF, a.causal_offset);
    x.put<int32_t>(FA_A64_OFF_ROPE_Q, a.rope_q ? 1 : 0);
    x.put<int32_t>(FA_A64_OFF_Q_ROPE_OFF, a.q_rope_offset);
    x.put<float>(FA_A64_OFF_C2, a.scale * 1.4426950408889634f);
    x.put<uint32_t>(FA_A64_OFF_NQB, nqb);
    x.put<uint32_t>(FA_A64_OFF_NB, nb);
    x.put<uint32_t>(FA_A64_OFF_GRID, wg);
    x.put<uint32_t>(FA_A64_OFF_UNITS, units);
    uint32_t m, sh;
    fastdiv(units, &m, &sh);
    x.put<uint32_t>(FA_A64_OFF_FD_UNITS_M, m);
    x.put<uint32_t>(FA_A64_OFF_FD_UNITS_S, sh);
    fastdiv((uint32_t)a.kv_heads, &m, &sh);
    x.put<uint32_t>(FA_A64_OFF_FD_KVH_M, m);
    x.put<uint32_t>(FA_A64_OFF_FD_KVH_S, sh);
    x.put<uint32_t>(FA_A64_OFF_ROPE_BYTES, a.rope_q ? (uint32_t)a.rope_rows * 512u : 0u);
    // byte extents of one (batch, kv head) slice of Q, O and LSE: the resource ranges
    const uint64_t g1 = (uint64_t)(a.group - 1), r1 = (uint64_t)(a.q_len - 1);
    x.put<uint32_t>(FA_A64_OFF_BATCH, (uint32_t)a.batch);
    x.put<uint32_t>(FA_A64_OFF_Q_NREC, (uint32_t)((g1 * a.q_sh + r1 * a.q_ss + 128) * 2));
    x.put<uint32_t>(FA_A64_OFF_O_NREC, (uint32_t)((g1 * a.o_sh + r1 * a.o_ss + 128) * 2));
    x.put<uint32_t>(FA_A64_OFF_LSE_NREC, (uint32_t)((g1 * a.lse_sh + r1 + 1) * 4));
    size_t bytes = sizeof x.b;
    void* extra[] = {HIP_LAUNCH_PARAM_BUFFER_POINTER, x.b, HIP_LAUNCH_PARAM_BUFFER_SIZE, &bytes,
                     HIP_LAUNCH_PARAM_END};
    hipFunction_t fn = current_fn(paged, a.k_lo != nullptr, dt == Dtype::F16);
    if (!fn) return;  // prefill_a64_eligible() checked this before the launch was chosen
    if (a.ev_start && a.ev_stop)
        (void)hipExtModuleLaunchKernel(fn, wg * 256, 1, 1, 256, 1, 1, 0, s, nullptr, extra,
                                       a.ev_start, a.ev_stop, 0);
    else
        (void)hipModuleLaunchKernel(fn, wg, 1, 1, 256, 1, 1, 0, s, nullptr, extra);
}

}  // namespace fa
