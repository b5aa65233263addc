// Token ids of texts without a checkpoint's tokenizer (host C++, C ABI): a word's or mark's id is its CRC-32's place among the
// ordinary ids.  32 captions of up to 132 words, ids and mask, took the interpreter 2.4 ms in a container of 8 CPUs, in front of
// 4.1 ms of an encoder's kernels; here 0.06.  One text of 32: 37 us and 19.
#include <algorithm>
#include <array>
#include <cstdint>
#include <vector>

namespace {

std::array<uint32_t, 256> crc_table() {
  std::array<uint32_t, 256> t;
  for (uint32_t i = 0; i < 256; ++i) {
    uint32_t c = i;
    for (int k = 0; k < 8; ++k) c = (c >> 1) ^ (c & 1 ? 0xEDB88320u : 0u);
    t[i] = c;
  }
  return t;
}

enum Kind : uint8_t { kSpace, kWord, kMark };

// of an ASCII character, as Python's regular expressions on str have it: 0x1c .. 0x1f are spaces too
std::array<Kind, 128> kinds() {
  std::array<Kind, 128> k;
  for (int c = 0; c < 128; ++c) {
    const bool word = (c >= '0' && c <= '9') || (c >= 'A' && c <= 'Z') || (c >= 'a' && c <= 'z') || c == '_';
    k[c] = word ? kWord : (c == ' ' || (c >= 9 && c <= 13) || (c >= 28 && c <= 31)) ? kSpace : kMark;
  }
  return k;
}

}  // namespace

extern "C" {

// text: the rows one after the other, ASCII; ends[r]: where row r ends.  ids, mask [rows, width]: ``bos`` (unless the row begins with
// it), the words, ``eos``; a row longer than ``width`` keeps width - 1 of it and eos, or its first width without an eos; ``pad`` behind.
// bos, eos: -1 for none.  Returns the longest row's length.
int shai_hash_rows(const uint8_t* text, const int64_t* ends, int rows, int first, int span, int bos, int eos, int pad, int width,
                   int64_t* ids, int64_t* mask) {
  static const std::array<uint32_t, 256> table = crc_table();
  static const std::array<Kind, 128> kind = kinds();
  int longest = 0;
  std::vector<int64_t> row;
  for (int r = 0; r < rows; ++r) {
    row.clear();
    const int64_t end = ends[r];
    // one more than fits says that the row is too long
    for (int64_t i = r ? ends[r - 1] : 0; i < end && (int64_t)row.size() <= width;) {
      const Kind k = kind[text[i] & 127];
      if (k == kSpace) {
        ++i;
        continue;
      }
      uint32_t c = 0xffffffffu;
      do {
        const uint8_t ch = text[i] >= 'A' && text[i] <= 'Z' ? text[i] + 32 : text[i];
        c = table[(c ^ ch) & 255] ^ (c >> 8);
        ++i;
      } while (k == kWord && i < end && kind[text[i] & 127] == kWord);
      row.push_back(first + (int64_t)((c ^ 0xffffffffu) % (uint32_t)span));
    }
    if (bos >= 0 && (row.empty() || row[0] != bos)) row.insert(row.begin(), bos);
    if (eos >= 0) row.push_back(eos);
    if ((int64_t)row.size() > width) {
      row.resize(width);
      if (eos >= 0) row[width - 1] = eos;
    }
    const int n = (int)row.size();
    longest = std::max(longest, n);
    int64_t* out = ids + (int64_t)r * width;
    std::copy(row.begin(), row.end(), out);
    std::fill(out + n, out + width, (int64_t)pad);
    std::fill(mask + (int64_t)r * width, mask + (int64_t)r * width + n, (int64_t)1);
    std::fill(mask + (int64_t)r * width + n, mask + (int64_t)(r + 1) * width, (int64_t)0);
  }
  return longest;
}

}  // extern "C"
