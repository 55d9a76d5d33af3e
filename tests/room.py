"""Processes that take room on a GPU's account (room_holder.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def build(folder):
    exe = os.path.join(str(folder), "room_holder")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-o", exe,
                    os.path.join(HERE, "room_holder.cpp")], check=True)
    return exe


class Holder:
    def __init__(self, exe, bus, units):
        self.p = subprocess.Popen([exe, bus, str(units)], stdin=subprocess.PIPE, stdout=subprocess.PIPE, text=True,
                                  bufsize=1)
        assert self.p.stdout.readline() == "open\n"

    def _ask(self, line):
        self.p.stdin.write(line + "\n")
        return self.p.stdout.readline() == "1\n"

    def take(self, n):
        return self._ask("take %d" % n)

    def give(self, n):
        assert self._ask("give %d" % n)

    def end(self, kill=False):
        if kill:
            self.p.kill()
        else:
            self.p.stdin.close()
        self.p.wait(timeout=20)
        self.p.stdout.close()
