// choices.cpp -- prints the kernel each call runs on, from the host-only rules the
// library's launchers use. Lines on stdin:
//   gemm M N K f32|f16 kn|nk [unaligned]   -> e.g. "256x128 SHIFT split" or "fp32 direct"
//   few N K                                -> "few_rows 48" (weight rows per workgroup) or "stream-K"
// The CU count is the first argument.
#include "gemm_choice.hpp"

#include <cstdlib>
#include <iostream>
#include <sstream>
#include <string>

int main(int argc, char** argv) {
  if (argc != 2) return 2;
  const long long cus = std::atoll(argv[1]);
  std::string line;
  while (std::getline(std::cin, line)) {
    std::istringstream in(line);
    std::string what;
    in >> what;
    if (what == "gemm") {
      eng::GemmShape s;
      std::string b, layout, aligned;
      in >> s.M >> s.N >> s.K >> b >> layout >> aligned;
      s.half_b = b == "f16";
      s.b_nk = layout == "nk";
      s.a16 = s.b16 = aligned != "unaligned";
      const eng::Fp32Choice fp32 = eng::gemm_fp32_choice(s, cus);
      const eng::SplitChoice c = eng::gemm_split_choice(s, cus);
      if (fp32.us <= c.cut.us) {
        const char* names[] = {"small", "direct", "staged"};
        std::cout << "fp32 " << names[static_cast<int>(fp32.kernel)] << "\n";
      } else {
        const char* forms[] = {"ALIGNED", "ANY", "SHIFT"};
        std::cout << c.bm << "x" << c.bn << " " << forms[eng::gemm_split_form(s)]
                  << (c.cut.split > 0 ? " split" : "") << "\n";
      }
    } else if (what == "few") {
      long long N = 0, K = 0;
      in >> N >> K;
      if (eng::few_rows_ahead(N, K, cus))
        std::cout << "few_rows " << 16 * eng::few_of(N, K, cus).rt << "\n";
      else
        std::cout << "stream-K\n";
    } else {
      return 2;
    }
  }
}
