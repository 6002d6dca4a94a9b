// Python module `neoGEMM`: the PyTorch-ROCm face of libneogemm.so.
//
// Keeps the reference's extension surface — module neoGEMM, function neoGemmV1(A, B, C) with keyword
// names A, B, C returning None (nemgemmV03.cu:343-399, neogemmv4.cu:335-338), the older
// neogemm(A, B, C) (v01.cu:272-317, neogemmV02.cu:304-307) — and adds C = gemm(A, B).  This file
// only unwraps tensors, checks them and calls the C ABI of include/neogemm.h on torch's current HIP
// stream; there is no kernel code and no HIP call here apart from asking torch for that stream.
//
// Differences from the reference launcher, on purpose:
//  * arguments are validated (the reference only checks dtype through data_ptr<>, nemgemmV03.cu:349-351)
//    and failures raise instead of printing to stderr (nemgemmV03.cu:387-390);
//  * the launch goes to torch's current stream, not the legacy default stream (nemgemmV03.cu:383);
//  * no state tied to a tensor is cached between calls (the reference caches TMA descriptors keyed on shape
//    only, nemgemmV03.cu:27-30,359-371, which goes stale when another tensor of the same shape is passed); the
//    only state kept is a scratch buffer of at most 64 MiB per (device, stream), for split-K partials and copies onto the 16-byte grid.
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <torch/extension.h>

#include <map>
#include <string>

#include "neogemm.h"

namespace {

void check_operand(const torch::Tensor& t, const char* name) {
  TORCH_CHECK(t.defined(), name, " is undefined");
  TORCH_CHECK(t.is_cuda(), name, " must be a GPU tensor");
  TORCH_CHECK(t.scalar_type() == at::kBFloat16, name, " must be bfloat16, got ", t.scalar_type());
  TORCH_CHECK(t.dim() == 2, name, " must be 2-D, got ", t.dim(), "-D");
}

// A 2-D tensor whose rows are contiguous (stride(1) == 1) is passed with ld = stride(0).
bool row_major(const torch::Tensor& t) { return t.size(1) <= 1 || t.stride(1) == 1; }
int64_t row_ld(const torch::Tensor& t) { return t.size(0) <= 1 ? std::max<int64_t>(t.size(1), 1) : t.stride(0); }

// Scratch of a call (split-K partials, copies of operands), one buffer per (device, stream): two GEMMs on two streams of one device
// must not share their partials, and a buffer is only ever used on the stream that was current when the caching allocator handed it out,
// which is the stream whose order the allocator follows when the block is reused.  So dropping a buffer that has
// become too small is safe: its block goes back to that stream's pool and is handed out again only to work queued
// on that same stream, behind the kernels that still use it.  The cache is per host thread.
// Two kinds of call take a block of their own from the caching allocator instead, and give it back when they return:
//  * one that is captured into a graph: the block comes from the graph's own memory then and stays valid for as long as the graph,
//    while a kept buffer that is outgrown later would be freed under the address that the graph replays;
//  * one that needs more than kMaxKept: it runs long enough not to notice, and nothing of that size stays behind it.
struct WorkspaceKey {
  int device;
  hipStream_t stream;
  bool operator<(const WorkspaceKey& o) const { return device != o.device ? device < o.device : stream < o.stream; }
};
// At most kMaxWorkspaces buffers are kept: streams come and go, and a buffer whose stream is gone would otherwise stay
// for the life of the thread.  The least recently used one is dropped (safe for the reason above).
constexpr size_t kMaxWorkspaces = 16;
constexpr size_t kMaxKept = (size_t)64 << 20;
struct WorkspaceSlot {
  torch::Tensor buffer;
  uint64_t last_use = 0;
};
torch::Tensor workspace_for(const torch::Tensor& like, hipStream_t stream, size_t bytes) {
  const auto options = like.options().dtype(torch::kUInt8);
  if (bytes > kMaxKept || c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None)
    return torch::empty({(int64_t)bytes}, options);
  static thread_local std::map<WorkspaceKey, WorkspaceSlot> ws;
  static thread_local uint64_t clock = 0;
  const WorkspaceKey key{(int)like.get_device(), stream};
  if (ws.find(key) == ws.end() && ws.size() >= kMaxWorkspaces) {
    auto oldest = ws.begin();
    for (auto it = ws.begin(); it != ws.end(); ++it)
      if (it->second.last_use < oldest->second.last_use) oldest = it;
    ws.erase(oldest);
  }
  WorkspaceSlot& slot = ws[key];
  slot.last_use = ++clock;
  torch::Tensor& t = slot.buffer;
  if (!t.defined() || (size_t)t.numel() < bytes) {
    t = torch::Tensor();  // give the old block back first
    t = torch::empty({(int64_t)bytes}, options);
  }
  return t;
}

// How many problems of one shape a call holds and how far apart they lie, in elements.
struct Batch {
  int64_t count = 1, sa = 0, sb = 0, sc = 0;
};
void run(const torch::Tensor& A, const torch::Tensor& B, torch::Tensor& C, int64_t M, int64_t N, int64_t K,
         int64_t lda, int64_t ldb, int64_t ldc, int a_layout, int b_layout, int c_layout, float alpha = 1.f, float beta = 0.f,
         const Batch& bt = Batch()) {
  // PyTorch-ROCm names its HIP devices "cuda"; these are the guard and stream accessors for that naming
  c10::hip::HIPGuardMasqueradingAsCUDA guard(A.device());
  const size_t need = neogemm_bf16_call_workspace_bytes(A.data_ptr(), B.data_ptr(), M, N, K, lda, ldb, a_layout, b_layout, c_layout, bt.sa,
                                                        bt.sb, bt.count);
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(A.get_device()).stream();
  const torch::Tensor scratch = need ? workspace_for(A, stream, need) : torch::Tensor();
  void* ws = need ? scratch.data_ptr() : nullptr;
  const int st = neogemm_bf16_general(A.data_ptr(), B.data_ptr(), C.data_ptr(), M, N, K, lda, ldb, ldc, a_layout, b_layout, c_layout,
                                      alpha, beta, bt.sa, bt.sb, bt.sc, bt.count, ws, need, (void*)stream);
  TORCH_CHECK(st == NEOGEMM_OK, "neogemm_bf16 failed: ", neogemm_strerror(st));
}

// How the two operands of a product lie in memory; a tensor that no layout describes is made contiguous.
struct Operands {
  torch::Tensor A, B;
  int a_layout = NEOGEMM_A_MK, b_layout = NEOGEMM_B_KN;
  int64_t lda, ldb;
};
// Whether the bytes from the first to the last element of a strided tensor meet those of another one.
bool overlap(const torch::Tensor& a, const torch::Tensor& b) {
  auto end = [](const torch::Tensor& t) {
    int64_t n = 1;
    for (int64_t d = 0; d < t.dim(); ++d) n += (t.size(d) - 1) * t.stride(d);
    return (uintptr_t)t.data_ptr() + n * t.element_size();
  };
  return a.numel() > 0 && b.numel() > 0 && (uintptr_t)a.data_ptr() < end(b) && (uintptr_t)b.data_ptr() < end(a);
}
// out: the tensor that is written while A and B are read (none: a new one).
Operands describe(torch::Tensor A, torch::Tensor B, const torch::Tensor* out = nullptr) {
  Operands o;
  if (row_major(B)) {
    o.ldb = row_ld(B);
  } else if (B.stride(0) == 1) {  // B = W.t() with W [N,K] row-major
    o.b_layout = NEOGEMM_B_NK;
    o.ldb = B.size(1) <= 1 ? std::max<int64_t>(B.size(0), 1) : B.stride(1);
  } else {
    B = B.contiguous();
    o.ldb = row_ld(B);
  }
  // A = X.t() with X [K,M] row-major, as in a weight gradient dY.t() * X, is read in place: by the tile kernels where it comes in
  // whole 16-byte chunks (a copy took 68 us for 4096 x 4096 where the product itself takes 98), by the kernel for operands at any
  // address where not.  A copy is made for the decode kernels, which want K-contiguous rows and few of them, and where C lies in A's
  // own memory (C = C.t() * X + C): a tile is read by workgroups that run after the one which has stored it.
  auto chunks = [](const torch::Tensor& t, int64_t ld) { return ((uintptr_t)t.data_ptr() & 15) == 0 && ld % 8 == 0; };
  const int64_t M = A.size(0), N = B.size(1), K = A.size(1);
  o.lda = row_ld(A);
  if (!row_major(A)) {
    const bool b_whole = chunks(B, o.ldb) && (o.b_layout == NEOGEMM_B_NK || N % 8 == 0);
    const bool decode = M <= 128 && K % 8 == 0 && b_whole;
    if (A.stride(0) == 1 && A.stride(1) >= M && !decode && !(out && overlap(A, *out))) {
      o.a_layout = NEOGEMM_A_KM;
      o.lda = A.stride(1);
    } else {
      A = A.contiguous();
      o.lda = row_ld(A);
    }
  }
  o.A = A;
  o.B = B;
  return o;
}

// C = gemm(A, B): A [M,K], B [K,N] -> new C [M,N], all bf16.  A transposed view of a contiguous
// tensor is taken as is where the kernels can read it (for B that is the reference's own layout).
torch::Tensor gemm(torch::Tensor A, torch::Tensor B) {
  check_operand(A, "A");
  check_operand(B, "B");
  TORCH_CHECK(A.device() == B.device(), "A and B must be on the same device");
  TORCH_CHECK(A.size(1) == B.size(0), "inner dimensions differ: A is ", A.sizes(), ", B is ", B.sizes());
  const int64_t M = A.size(0), K = A.size(1), N = B.size(1);
  torch::Tensor C = torch::empty({M, N}, A.options());
  if (M == 0 || N == 0) return C;
  const Operands o = describe(std::move(A), std::move(B));
  run(o.A, o.B, C, M, N, K, o.lda, o.ldb, std::max<int64_t>(N, 1), o.a_layout, o.b_layout, NEOGEMM_C_ROW);
  return C;
}

// gemm_scaled(A, B, C, alpha, beta): C[M,N] (row-major, contiguous) = alpha * A[M,K] @ B[K,N] + beta * C, in place;
// the epilogue the reference's v4 kernel declares (neogemmv4.cu:166,266).
void gemm_scaled(torch::Tensor A, torch::Tensor B, torch::Tensor C, double alpha, double beta) {
  check_operand(A, "A");
  check_operand(B, "B");
  check_operand(C, "C");
  TORCH_CHECK(A.device() == B.device() && A.device() == C.device(), "A, B and C must be on the same device");
  TORCH_CHECK(A.size(1) == B.size(0), "inner dimensions differ: A is ", A.sizes(), ", B is ", B.sizes());
  TORCH_CHECK(C.size(0) == A.size(0) && C.size(1) == B.size(1) && C.is_contiguous(), "C must be a contiguous [M,N]");
  const int64_t M = A.size(0), K = A.size(1), N = B.size(1);
  if (M == 0 || N == 0) return;
  const Operands o = describe(std::move(A), std::move(B), &C);
  run(o.A, o.B, C, M, N, K, o.lda, o.ldb, std::max<int64_t>(N, 1), o.a_layout, o.b_layout, NEOGEMM_C_ROW, (float)alpha, (float)beta);
}

// bmm(A, B): A [b,M,K], B [b,K,N] or [K,N] (shared) -> new C [b,M,N]; one launch (neogemm_bf16_general).  Either operand may be
// a transposed view (the k^T of attention scores) or a slice of a larger tensor: it is read in place unless only a copy of it would
// lie on the 16-byte grid.
torch::Tensor bmm(torch::Tensor A, torch::Tensor B) {
  TORCH_CHECK(A.is_cuda() && B.is_cuda(), "A and B must be GPU tensors (there is no CPU path)");
  TORCH_CHECK(A.scalar_type() == torch::kBFloat16 && B.scalar_type() == torch::kBFloat16, "A and B must be bfloat16");
  TORCH_CHECK(A.dim() == 3 && (B.dim() == 3 || B.dim() == 2), "A must be [b,M,K], B [b,K,N] or [K,N]");
  TORCH_CHECK(A.device() == B.device(), "A and B must be on the same device");
  TORCH_CHECK(A.size(2) == B.size(B.dim() - 2) && (B.dim() == 2 || B.size(0) == A.size(0)), "shapes do not match: A ",
              A.sizes(), ", B ", B.sizes());
  const int64_t batch = A.size(0), M = A.size(1), K = A.size(2), N = B.size(B.dim() - 1);
  torch::Tensor C = torch::empty({batch, M, N}, A.options());
  if (batch == 0 || M == 0 || N == 0) return C;
  // rows x cols matrices of a 3-D tensor: row-major or its transpose, and the leading dimension
  struct View {
    bool ok, transposed;
    int64_t ld, stride;
    bool whole;  // on the 16-byte grid
  };
  auto view = [](const torch::Tensor& t) -> View {
    const int d = t.dim() - 2;
    const int64_t rows = t.size(d), cols = t.size(d + 1), sr = t.stride(d), sc = t.stride(d + 1);
    View v{true, false, std::max<int64_t>(cols, 1), d && t.size(0) > 1 ? t.stride(0) : 0, false};
    if (cols <= 1 || sc == 1) {
      if (rows > 1) v.ld = sr;
      v.ok = v.ld >= cols;
    } else if (rows <= 1 || sr == 1) {
      v.transposed = true;
      v.ld = sc;
      v.ok = sc >= rows;
    } else {
      v.ok = false;
    }
    v.whole = ((uintptr_t)t.data_ptr() & 15) == 0 && v.ld % 8 == 0 && v.ld < (1 << 21) && v.stride % 8 == 0 && (v.transposed ? rows : cols) % 8 == 0;
    return v;
  };
  auto settle = [&](torch::Tensor& t) -> View {
    View v = view(t);
    if (t.is_contiguous() || (v.ok && (v.whole || t.size(t.dim() - 1) % 8 != 0))) return v;
    t = t.contiguous();
    return view(t);
  };
  if (batch == 1 && M <= 128 && A.stride(2) != 1) A = A.contiguous();  // the decode kernels want K-contiguous rows
  const View va = settle(A), vb = settle(B);
  run(A, B, C, M, N, K, va.ld, vb.ld, std::max<int64_t>(N, 1), va.transposed ? NEOGEMM_A_KM : NEOGEMM_A_MK,
      vb.transposed ? NEOGEMM_B_NK : NEOGEMM_B_KN, NEOGEMM_C_ROW, 1.f, 0.f, Batch{batch, va.stride, vb.stride, M * N});
  return C;
}

// neoGemmV1(A, B, C): A [M,K], B [N,K], C holds M*N bf16 and receives the product column-major,
// so that C.t() (viewing the [M,N]-shaped C of benchmark.py:12 transposed, benchmark.py:25) equals
// A @ B.t() (benchmark.py:18) when M == N, and C.view(N, M).t() does in general.
void neoGemmV1(torch::Tensor A, torch::Tensor B, torch::Tensor C) {
  check_operand(A, "A");
  check_operand(B, "B");
  check_operand(C, "C");
  TORCH_CHECK(A.device() == B.device() && A.device() == C.device(), "A, B and C must be on the same device");
  TORCH_CHECK(A.size(1) == B.size(1), "A is [M,K] and B is [N,K]: K differs (", A.size(1), " vs ", B.size(1), ")");
  TORCH_CHECK(A.is_contiguous() && B.is_contiguous() && C.is_contiguous(), "A, B and C must be contiguous");
  const int64_t M = A.size(0), K = A.size(1), N = B.size(0);
  TORCH_CHECK(C.numel() == M * N, "C must hold M*N = ", M * N, " elements, has ", C.numel());
  if (M == 0 || N == 0) return;
  run(A, B, C, M, N, K, std::max<int64_t>(K, 1), std::max<int64_t>(K, 1), M, NEOGEMM_A_MK, NEOGEMM_B_NK, NEOGEMM_C_COL);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "BF16 GEMM for MI355X (gfx950): bf16 in, fp32 accumulate, bf16 out";
  m.def("gemm", &gemm, "C[M,N] = A[M,K] @ B[K,N]", py::arg("A"), py::arg("B"));
  m.def("neoGemmV1", &neoGemmV1, "C (column-major) = A[M,K] @ B[N,K]^T, in place", py::arg("A"), py::arg("B"),
        py::arg("C"));
  m.def("neogemm", &neoGemmV1, "alias of neoGemmV1 (the reference's first module name)", py::arg("A"),
        py::arg("B"), py::arg("C"));
  m.def("gemm_scaled", &gemm_scaled, "C = alpha * A[M,K] @ B[K,N] + beta * C, in place", py::arg("A"), py::arg("B"),
        py::arg("C"), py::arg("alpha") = 1.0, py::arg("beta") = 0.0);
  m.def("bmm", &bmm, "C[b,M,N] = A[b,M,K] @ B[b,K,N] (or B [K,N] shared)", py::arg("A"), py::arg("B"));
  m.def("version", []() { return std::string(neogemm_version()); });
}
