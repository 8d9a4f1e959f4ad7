// String helpers and the error-message convention of the reference
// (src/errors.h:7-12, src/utils.h:14-36).
#ifndef QFLEX_AMD_UTILS_H_
#define QFLEX_AMD_UTILS_H_

#include <sstream>
#include <string>
#include <string_view>
#include <type_traits>

namespace qflex::utils {

// x as an output stream writes it, behind `out` (no stream for strings and
// whole numbers: index names are made of them, hundreds per circuit).
template <typename T>
void append(std::string& out, const T& x) {
  if constexpr (std::is_same_v<T, char> || std::is_same_v<T, signed char> ||
                std::is_same_v<T, unsigned char>) {
    out.push_back(char(x));
  } else if constexpr (std::is_convertible_v<const T&, std::string_view>) {
    out.append(std::string_view(x));
  } else if constexpr (std::is_integral_v<T>) {
    out += std::to_string(x);
  } else {
    std::ostringstream ss;
    ss << x;
    out += ss.str();
  }
}

template <typename... T>
std::string concat(const T&... x) {
  std::string out;
  (append(out, x), ...);
  return out;
}

// "Thu Aug 23 14:55:02 2001"
std::string get_date_time();

// "1GB" / "512 MB" / "1024" -> bytes (suffixes GB, MB, KB, B; 1024-based).
std::size_t from_readable_memory_string(std::string memory);

// bytes -> "6.26 GB" (two decimals, 1024-based).
std::string readable_memory_string(double memory);

}  // namespace qflex::utils

#endif
