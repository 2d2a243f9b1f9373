// MmapFile for test_metal_ops where no reference checkout was built: the class
// is declared by include/lite_ssm/allocator.hpp and is the application's own in
// a program that links this backend.
#include <fcntl.h>
#include <sys/mman.h>
#include <sys/stat.h>
#include <unistd.h>

#include <stdexcept>

#include "lite_ssm/allocator.hpp"

namespace lite_ssm {

MmapFile::MmapFile(const std::string& path) {
    const int fd = open(path.c_str(), O_RDONLY | O_CLOEXEC);
    struct stat st {};
    if (fd >= 0 && fstat(fd, &st) == 0 && st.st_size > 0) {
        file_size_ = static_cast<std::size_t>(st.st_size);
        const std::size_t page = static_cast<std::size_t>(sysconf(_SC_PAGESIZE));
        mapped_size_ = (file_size_ + page - 1) / page * page;
        void* p = mmap(nullptr, mapped_size_, PROT_READ, MAP_PRIVATE, fd, 0);
        if (p != MAP_FAILED) ptr_ = p;
    }
    if (fd >= 0) close(fd);
    if (!ptr_) throw std::runtime_error("cannot map " + path);
}

MmapFile::~MmapFile() {
    if (ptr_) munmap(ptr_, mapped_size_);
}

}  // namespace lite_ssm
