// Turns of processes that share a GPU (ranks of one job, say): an flock on an
// empty file named after the GPU, taken around a launch whose workgroups wait for
// each other. Two such launches at once could each hold CUs that the other needs.
// The lock goes with the process that holds it, however that ends. Processes that
// do not see each other's files (other containers) are not ordered by it: their
// launches rely on the limit of their own waits.
#include <errno.h>
#include <fcntl.h>
#include <sys/file.h>
#include <time.h>
#include <unistd.h>

#include <string>

namespace bhip {

// The file, open for locking, in the first of the directories that allows it; -1
// if none does. (Opened without creating it first: a file of another user in a
// directory with the sticky bit must not be opened with O_CREAT.)
static int turn_open(const char* const* dirs, int ndirs, const std::string& name) {
  for (int i = 0; i < ndirs; ++i) {
    const std::string path = std::string(dirs[i]) + "/" + name;
    const int flags = O_RDONLY | O_CLOEXEC | O_NOFOLLOW;
    int fd = open(path.c_str(), flags);
    if (fd < 0 && errno == ENOENT) fd = open(path.c_str(), flags | O_CREAT | O_EXCL, 0644);
    if (fd < 0 && errno == EEXIST) fd = open(path.c_str(), flags);  // made just now by another
    if (fd >= 0) return fd;
  }
  return -1;
}

// Takes the turn, waiting for at most `limit` seconds: false if another process
// has had it for that long. True without a file, or where locks do not work.
static bool turn_take(int fd, double limit) {
  if (fd < 0) return true;
  timespec t0, t;
  clock_gettime(CLOCK_MONOTONIC, &t0);
  for (;;) {
    if (flock(fd, LOCK_EX | LOCK_NB) == 0) return true;
    if (errno == EINTR) continue;
    if (errno != EWOULDBLOCK) return true;
    clock_gettime(CLOCK_MONOTONIC, &t);
    if ((double)(t.tv_sec - t0.tv_sec) + 1e-9 * (double)(t.tv_nsec - t0.tv_nsec) >= limit)
      return false;
    const timespec nap = {0, 20000};
    nanosleep(&nap, nullptr);
  }
}

static void turn_give(int fd) {
  if (fd >= 0) (void)flock(fd, LOCK_UN);
}

}  // namespace bhip
