// Turns of processes (argument: a directory). Prints "ok" or what is wrong.
#include "turn.inl"

#include <signal.h>
#include <stdio.h>
#include <sys/stat.h>
#include <sys/wait.h>

using namespace bhip;

static int wrong(const char* what) {
  printf("%s\n", what);
  return 1;
}
static double now() {
  timespec t;
  clock_gettime(CLOCK_MONOTONIC, &t);
  return (double)t.tv_sec + 1e-9 * (double)t.tv_nsec;
}

int main(int, char** argv) {
  const std::string none = std::string(argv[1]) + "/absent";
  const char* dirs[] = {none.c_str(), argv[1]};
  if (turn_open(dirs, 1, "gpu") >= 0) return wrong("opened in a directory that is not there");
  if (!turn_take(-1, 0.0)) return wrong("no file, no turn");
  turn_give(-1);
  // a link in the file's place is not followed
  if (symlink("elsewhere", (std::string(argv[1]) + "/link").c_str())) return wrong("symlink");
  if (turn_open(dirs, 2, "link") >= 0) return wrong("followed a link");
  const int fd = turn_open(dirs, 2, "gpu");
  if (fd < 0) return wrong("not opened");
  if (!turn_take(fd, 0.0)) return wrong("free, but not taken");
  turn_give(fd);
  // another process has it, until it is killed
  int up[2];
  if (pipe(up)) return wrong("pipe");
  const pid_t child = fork();
  if (child == 0) {
    const int mine = turn_open(dirs, 2, "gpu");
    char c = turn_take(mine, 0.0) ? 'y' : 'n';
    if (write(up[1], &c, 1) != 1) _exit(1);
    for (;;) pause();
  }
  char c = 0;
  if (read(up[0], &c, 1) != 1 || c != 'y') return wrong("child");
  const double t0 = now();
  if (turn_take(fd, 0.05)) return wrong("taken twice");
  const double waited = now() - t0;
  if (waited < 0.05 || waited > 2.0) return wrong("limit");
  kill(child, SIGKILL);
  if (!turn_take(fd, 20.0)) return wrong("not free after its process ended");
  waitpid(child, nullptr, 0);
  turn_give(fd);
  // processes that add to a number each in its turn
  FILE* f = fopen((std::string(argv[1]) + "/count").c_str(), "w+");
  const int zero = 0;
  fwrite(&zero, sizeof zero, 1, f);
  fclose(f);
  for (int p = 0; p < 4; ++p)
    if (fork() == 0) {
      const int mine = turn_open(dirs, 2, "gpu");
      const int at = open((std::string(argv[1]) + "/count").c_str(), O_RDWR);
      for (int i = 0; i < 200; ++i) {
        if (!turn_take(mine, 60.0)) _exit(1);
        int v = 0;
        if (pread(at, &v, sizeof v, 0) != sizeof v) _exit(1);
        ++v;
        if (pwrite(at, &v, sizeof v, 0) != sizeof v) _exit(1);
        turn_give(mine);
      }
      _exit(0);
    }
  for (int p = 0, st = 0; p < 4; ++p)
    if (wait(&st) < 0 || st != 0) return wrong("a process failed");
  int v = 0;
  f = fopen((std::string(argv[1]) + "/count").c_str(), "r");
  if (!f || fread(&v, sizeof v, 1, f) != 1 || v != 800) return wrong("not in turns");
  printf("ok\n");
  return 0;
}
