// CPU checks of the GEMM planner (runtime.cpp, included whole: the planner is
// file-local). Reads one command per line, answers one line; nothing here
// touches a device.
//
//   plan M N K a_kc b_kc epi lda ldb permA permB   "<kernel> <slices>" or "refused"
//   apart (the same)                                of a product whose partials a launch of its own sums
//   beside (the same)                               of a layer's gradients that are to share a launch
//   pair (the same)                                 of one of two such problems in a launch
//   names                                           every kernel's name on one line
//   scratch M N K                                   "<floats reserved for up to K rows> <most that any takes>"
#include "../zealot_amd/csrc/runtime/runtime.cpp"

#include <cstdio>
#include <iostream>
#include <sstream>

namespace zl {  // of noalloc.hip, not reached here
void noalloc_setup(zl_ctx*) {}
void noalloc_release(zl_ctx*) {}
}  // namespace zl
using namespace zl;

static zl_status plan(zl_ctx& c, int M, int N, int K, bool a_kc, bool b_kc, int epi, int lda, int ldb, bool pa, bool pb,
                      const std::string& how, GemmPlan& P) {
  alignas(16) static float mem[4];
  static int perm[4];
  GemmDesc d;
  d.A = d.B = d.bias = d.Y = mem;
  d.C = mem;
  d.a_kc = a_kc;
  d.b_kc = b_kc;
  d.M = M;
  d.N = N;
  d.K = K;
  d.lda = lda;
  d.ldb = ldb;
  d.ldc = d.ldy = (int)round_up(N, 4);
  d.epi = epi;
  d.permA = pa ? perm : nullptr;
  d.permB = pb ? perm : nullptr;
  zk::ReduceSeg seg;
  d.seg_out = how == "apart" ? nullptr : &seg;
  d.beside = how == "beside";
  return plan_gemm(&c, d, P, how == "pair" ? 2 * cdiv(M, 128) * cdiv(N, 128) : 0);
}

int main() {
  zl_ctx c;
  std::string line, cmd;
  while (std::getline(std::cin, line)) {
    std::istringstream in(line);
    in >> cmd;
    if (cmd == "plan" || cmd == "apart" || cmd == "beside" || cmd == "pair") {
      int M, N, K, a, b, epi, lda, ldb, pa, pb;
      in >> M >> N >> K >> a >> b >> epi >> lda >> ldb >> pa >> pb;
      GemmPlan P;
      if (plan(c, M, N, K, a, b, epi, lda, ldb, pa, pb, cmd, P))
        std::puts("refused");
      else
        std::printf("%s %d\n", kGemmTable[P.kid - K_GEMM_BASE].name, P.splits);
    } else if (cmd == "names") {
      for (int k = 0; k < K_GEMM_BASE + kGemmCount; ++k) std::printf("%s ", kernel_name(k));
      std::puts("");
    } else {  // a weight gradient's scratch, reserved for K rows and used for any up to K
      int M, N, K;
      in >> M >> N >> K;
      size_t most = 0;
      for (int k = 1; k <= K; ++k)
        for (int form = 0; form < 6; ++form) {
          static const char* const how[3] = {"plan", "apart", "beside"};
          GemmPlan P;
          const int pad = form & 1;  // rows that are not float4-aligned
          if (plan(c, M, N, k, false, false, zk::kEpiStore, (int)round_up(M, 4) + pad, (int)round_up(N, 4) + pad, false,
                   false, how[form / 2], P))
            continue;
          if (P.splits > 1) most = std::max(most, (size_t)P.splits * M * N + (size_t)P.splits * M);
        }
      std::printf("%zu %zu\n", gemm_ws_floats(&c, M, N, K, false, false, zk::kEpiStore), most);
    }
  }
}
