// How much of a GPU is taken by launches whose workgroups wait for one another
// (the coarse CG in one launch), for all processes of a user.
//
// A launch that waits must have all its workgroups on the chip.  Alone it may
// take all of it.  Beside others it may only bring the sum to half of the chip: a
// workgroup takes at most half a CU, so then some CU always has room for the
// next one, however the others lie.  Kernels that do not wait need no place
// here: they end.  A launch that finds no room is not made.
//
// The account is a board in POSIX shared memory, one per user and GPU (by its
// PCI address), with a line for each process.  A process holds its line by a
// lock on a byte of the board's file, which the system drops when the process
// ends in any way; what a line without a holder says is not counted.  Where
// there is no shared memory the account is the process's own, and a launch
// beside another process's may lose its waits, which are bounded.
#pragma once

#include <cerrno>
#include <cstdint>
#include <fcntl.h>
#include <mutex>
#include <pthread.h>
#include <string>
#include <sys/file.h>
#include <sys/mman.h>
#include <sys/stat.h>
#include <unistd.h>

namespace wavi {

constexpr int ROOM_LINES = 64;

struct RoomBoard {
    pthread_mutex_t mu;  // shared, robust
    int32_t laid_out;
    int32_t used[ROOM_LINES];
};

class Room {
public:
    // The account of the GPU at PCI address `bus` with room for `all` units.
    // Called once.
    void open(const char *bus, int all)
    {
        all_ = all;
        std::string name = "/wavi_hip_room1." + std::to_string((unsigned long)geteuid()) + ".";
        for (const char *c = bus; *c; ++c) name += *c == ':' || *c == '/' ? '-' : *c;
        fd_ = shm_open(name.c_str(), O_RDWR | O_CREAT | O_CLOEXEC, 0600);
        if (fd_ >= 0 && !attach()) {
            close(fd_);
            fd_ = -1;
        }
        if (fd_ < 0) {
            board_ = &own_;
            lay_out(PTHREAD_PROCESS_PRIVATE);
            line_ = 0;
        }
    }

    bool take(int units)
    {
        if (!board_ || line_ < 0 || !lock()) return false;
        bool ok = fits(units);
        if (!ok && drop_lines_without_holder()) ok = fits(units);
        if (ok) board_->used[line_] += units;
        pthread_mutex_unlock(&board_->mu);
        return ok;
    }

    void give(int units)
    {
        if (!board_ || line_ < 0 || !lock()) return;
        board_->used[line_] -= units;
        pthread_mutex_unlock(&board_->mu);
    }

private:
    RoomBoard own_ = {};
    RoomBoard *board_ = nullptr;
    int fd_ = -1, line_ = -1, all_ = 0;

    // Lock on byte k of the board's file; F_OFD_GETLK: whether another holds it.
    struct flock byte(int k) const
    {
        struct flock f = {};
        f.l_type = F_WRLCK;
        f.l_whence = SEEK_SET;
        f.l_start = k;
        f.l_len = 1;
        return f;
    }
    bool held(int k) const
    {
        struct flock f = byte(k);
        return fcntl(fd_, F_OFD_GETLK, &f) != 0 || f.l_type != F_UNLCK;
    }

    void lay_out(int shared)
    {
        pthread_mutexattr_t a;
        pthread_mutexattr_init(&a);
        pthread_mutexattr_setpshared(&a, shared);
        pthread_mutexattr_setrobust(&a, PTHREAD_MUTEX_ROBUST);
        pthread_mutex_init(&board_->mu, &a);
        pthread_mutexattr_destroy(&a);
        board_->laid_out = 1;
    }

    // Maps the board, lays it out if it is new, and takes a line of it.
    bool attach()
    {
        if (flock(fd_, LOCK_EX) != 0) return false;
        struct stat st;
        bool ok = fstat(fd_, &st) == 0 &&
                  (st.st_size >= (off_t)sizeof(RoomBoard) || posix_fallocate(fd_, 0, sizeof(RoomBoard)) == 0);
        if (ok) {
            void *p = mmap(nullptr, sizeof(RoomBoard), PROT_READ | PROT_WRITE, MAP_SHARED, fd_, 0);
            ok = p != MAP_FAILED;
            if (ok) board_ = (RoomBoard *)p;
        }
        if (ok) {
            if (!board_->laid_out) lay_out(PTHREAD_PROCESS_SHARED);
            for (int k = 0; k < ROOM_LINES && line_ < 0; ++k) {
                struct flock f = byte(k);
                if (fcntl(fd_, F_OFD_SETLK, &f) == 0) line_ = k;
            }
            // no line left: this process makes no launches that wait
            if (line_ >= 0 && lock()) {
                board_->used[line_] = 0;
                pthread_mutex_unlock(&board_->mu);
            }
        }
        (void)flock(fd_, LOCK_UN);
        return ok;
    }

    bool lock()
    {
        const int rc = pthread_mutex_lock(&board_->mu);
        if (rc == EOWNERDEAD) return pthread_mutex_consistent(&board_->mu) == 0;  // every line is one word
        return rc == 0;
    }

    bool fits(int units) const
    {
        int64_t used = 0;
        for (int k = 0; k < ROOM_LINES; ++k) used += board_->used[k];
        return used + units <= (used == 0 ? all_ : all_ / 2);
    }

    bool drop_lines_without_holder()
    {
        bool any = false;
        for (int k = 0; k < ROOM_LINES && fd_ >= 0; ++k)
            if (k != line_ && board_->used[k] != 0 && !held(k)) {
                board_->used[k] = 0;
                any = true;
            }
        return any;
    }
};

}  // namespace wavi
