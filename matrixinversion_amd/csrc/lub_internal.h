// lub_internal.h -- declarations shared by the kernel translation units and the
// C-ABI layer of liblubatch.so (not part of the public interface).
#pragma once

#include <stdint.h>

namespace lub {

constexpr int kMaxN = 32;
constexpr int kNumPivot = 5;   // NONE, PARALLEL, SERIAL, TREE, GEPP
constexpr int kNumLayout = 2;  // 0: 16 lanes per matrix (n <= 32), 1: 4 lanes per matrix (n <= 16)
constexpr int kLayoutLanes[kNumLayout] = {16, 4};
constexpr int kLayoutMaxN[kNumLayout] = {32, 16};

// Host handles of the launchable kernels, filled by the per-size-range
// translation units (each one instantiates lu_inverse_kernel<N, L, PIV> for
// its range of N and registers the host stubs here).
struct KernelTable {
  const void* plain[kMaxN + 1][kNumPivot][kNumLayout];
  // n % 4 == 0: the same kernels with the row padding flipped from its default
  const void* plain_flip[kMaxN + 1][kNumPivot][kNumLayout];
  const void* ragged[kNumPivot];
  // [layout]: inverse + one refinement step, and the step for a given inverse
  const void* refined[kMaxN + 1][kNumPivot][kNumLayout];
  const void* refine[kMaxN + 1][kNumLayout];
};

// Per-n launch choices shared by the plain and the ragged paths (set by the
// autotuner through lu_tuning_set, defaults in lub_api.hip).
struct Tuning {
  int8_t layout[kMaxN + 1];  // 0: 16-lane rows, 1: quads
  int8_t grab[kMaxN + 1];    // ragged: wave tiles per work item
  int8_t pad[kMaxN + 1];     // plain path, n % 4 == 0: LDS rows padded by 4 floats (1) or not (0)
};

// LDS row padding compiled into a kernel without the flip bit
// (Geo<N, L, V>::PAD for V & 2 == 0): rows of n % 8 == 0.
constexpr int8_t geo_pad(int n) { return (n > 0 && n % 8 == 0) ? 1 : 0; }
// Initial padding table of the plain path: every n % 4 == 0 but n = 28
// (measured on MI355X with the autotuner: padding n = 12 and n = 20 saves
// 4 % and 9 % of the kernel time, at n = 28 it costs 7 %).
constexpr int8_t initial_pad(int n) { return (n > 0 && n % 4 == 0 && n != 28) ? 1 : 0; }
Tuning current_tuning();

// Where the table's quads give way to 16-lane rows under LUB_LAYOUT_AUTO.
// Partial pivoting holds rows, and a quad's lane would hold three of them
// from n = 9 (four from n = 13): the pivot row's selection and its masked LDS
// stores then cost several times the update (100k matrices, quads / rows: n =
// 8 14 / 21 us, n = 9 85 / 25, n = 12 229 / 38, n = 16 514 / 59).  The other
// rules' chains are longer in quads too, which shows only while the chip is
// not full: 4,096 matrices of n = 12 4.9 / 3.9 us, 16,384 6.8 / 6.9, 100k
// 23 / 25.  The initial table has quads up to n = 12; one that has them above
// is taken at its word.
constexpr int kGeppQuadMaxN = 8;
constexpr int kSmallBatchMaxN = 12;
constexpr int64_t kSmallBatchQuads = 8192;
// The refined kernels take a quad tile's 16 matrices' steps one after the
// other, so their line lies higher (n = 12, 16,384 matrices: 13.3 / 10.3 us;
// 100k: 47.5 / 48.2).
constexpr int64_t kSmallBatchRefinedQuads = 16384;
constexpr bool rows_beat_quads(int n, bool gepp, int64_t batch, int64_t small_batch = kSmallBatchQuads) {
  return n > kGeppQuadMaxN && (gepp || (n <= kSmallBatchMaxN && batch <= small_batch));
}
// Layout of a call: the one that `flags` or LUB_LANES force, else rows where
// they beat quads, else the table's.
int choose_layout(int n, int flags, int64_t batch, int64_t small_batch = kSmallBatchQuads);

constexpr int kRefineQuadMaxN = 12;  // quads of the refinement of a given inverse
const KernelTable& kernel_table();

// Ragged batches of up to this many matrices run without a plan.
constexpr int64_t kRaggedDirectMax = 2048;

// The ragged inversion without a plan (batch <= kRaggedDirectMax, arguments
// checked).  The three arrays may be pinned host memory.  hdr (nullable): the
// planning header that receives the count of matrices with n outside 1..32.
// cus: the device's compute units (for ragged_persistent_grid).
int enqueue_ragged_direct(int* hdr, int cus, float* A, const int64_t* offsets, const int* ns, int* piv,
                          const int64_t* piv_offsets, int64_t batch, int flags, void* stream);

// The plain launch behind lu_batched_inverse_async64; info (nullable, one int
// per matrix) receives 0 or 1 + the first step with an exactly zero pivot.
int enqueue_plain(float* A, int* piv, int* info, int n, int64_t batch, int flags, void* stream);

}  // namespace lub

// One registration function per kernel translation unit.
#define LUB_REGISTER_DECL(lo, hi) extern "C" void lub_register_##lo##_##hi(lub::KernelTable* t)
LUB_REGISTER_DECL(1, 8);
LUB_REGISTER_DECL(9, 16);
LUB_REGISTER_DECL(17, 20);
LUB_REGISTER_DECL(21, 24);
LUB_REGISTER_DECL(25, 28);
LUB_REGISTER_DECL(29, 32);
extern "C" void lub_register_ragged_0(lub::KernelTable* t);
extern "C" void lub_register_ragged_1(lub::KernelTable* t);
extern "C" void lub_register_ragged_3(lub::KernelTable* t);
extern "C" void lub_register_ragged_4(lub::KernelTable* t);
extern "C" void lub_register_refined_1_8(lub::KernelTable* t);
extern "C" void lub_register_refined_9_12(lub::KernelTable* t);
extern "C" void lub_register_refined_13_18(lub::KernelTable* t);
extern "C" void lub_register_refined_19_23(lub::KernelTable* t);
extern "C" void lub_register_refined_24_27(lub::KernelTable* t);
extern "C" void lub_register_refined_28_30(lub::KernelTable* t);
extern "C" void lub_register_refined_31_32(lub::KernelTable* t);
